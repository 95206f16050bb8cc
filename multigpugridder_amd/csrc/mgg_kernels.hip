// HIP kernels for the Fourier-domain projection gridder, written for gfx950
// (CDNA4, wave64).
//
// Numerics contract.  This file is compiled with -ffp-contract=off, so every
// fused multiply-add is written explicitly (fmaf).  The FP32 expressions that
// feed discrete decisions (rotated coordinates, roundf of them, kernel-table
// indices, the mask and slab tests) follow the reference kernels as nvcc
// compiles them by default (--fmad=true; the reference's build passes no
// flags): a multiply feeding an add is contracted, without reassociation,
// each add of two products fusing its first operand:
//   a*x + b*y + c           -> fl(fma(a, x, fl(b*y)) + c)       (ref_sum2c)
//   x0*a0 + x1*a1 + x2*a2   -> fma(x2, a2, fma(x0, a0, fl(x1*a1)))  (ref_sum3)
//   r*kerScale + kerCenter  -> fma(r, kerScale, kerCenter)
// The CPU oracle restates the same reading, so rounding decisions match it
// bit for bit; accumulation order is free (FP32 here, FP64 in the oracle).
//
// Layout: column-major, x fastest.  vol[x + y*V + z*V*V];
// CAS image a: img[a*M*M + i + j*M]; a direction is 9 floats [u; v; n].
#include "mgg_columns.h"
#include "mgg_internal.h"

#include <hip/hip_fp16.h>

#include <algorithm>
#include <climits>
#include <type_traits>
#include <vector>

namespace mgg {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef unsigned int u4 __attribute__((ext_vector_type(4)));
typedef unsigned int u3 __attribute__((ext_vector_type(3)));

constexpr int kThreads = 256;

// ---------------------------------------------------------------------------
// Decision arithmetic as contracted by nvcc (see the numerics contract above).
// ---------------------------------------------------------------------------
// a*x + b*y + c: a pixel's rotated coordinate (gpuForwardProject.cu:53-55) or
// a back-projection tap position (gpuBackProject.cu:77,84,91).
__device__ __forceinline__ float ref_sum2c(float a, float x, float b, float y, float c)
{
    return fmaf(a, x, b * y) + c;
}
// x0*a0 + x1*a1 + x2*a2: a voxel's image-frame coordinate before its constant
// (gpuBackProject.cu:62-64).
__device__ __forceinline__ float ref_sum3(float x0, float a0, float x1, float a1, float x2, float a2)
{
    return fmaf(x2, a2, fmaf(x0, a0, x1 * a1));
}

// Kernel-table index (gpuForwardProject.cu:63-67, gpuBackProject.cu:79-82):
// clamp to [-convW, convW], scale and offset (one FMA), round half away from
// zero, clamp to table.
__device__ __forceinline__ int kb_index(float r, float fW, float kerScale, float kerCenter,
                                        int K)
{
    r = fminf(fmaxf(r, -fW), fW);
    const float s = fmaf(r, kerScale, kerCenter);
    int idx = (int)roundf(s);
    idx = min(max(idx, 0), K - 1);
    return idx;
}

// XCD-aware work mapping: hardware hands consecutive workgroup ids to the 8
// XCDs round-robin; remapping gives each XCD a contiguous run of work items so
// neighbouring tiles of one direction share that XCD's L2.
__device__ __forceinline__ unsigned xcd_work(unsigned perXcd)
{
    unsigned b = blockIdx.x;
    return (b & 7u) * perXcd + (b >> 3);
}

// ---------------------------------------------------------------------------
// Volume loads for the three storage types.  row5 fetches the 5 contiguous
// x-taps of one (y, z) row with unaligned vector loads.
// ---------------------------------------------------------------------------
template <int DT> struct VolLoad;

template <> struct VolLoad<DT_F32> {
    typedef float T;
    static constexpr int kRowSlack = 0;  // elements read past the 5th tap
    static __device__ __forceinline__ float one(const float *p) { return *p; }
    static __device__ __forceinline__ void row5(const float *p, float (&r)[5])
    {
        f4 a;
        __builtin_memcpy(&a, p, 16);
        r[0] = a.x; r[1] = a.y; r[2] = a.z; r[3] = a.w;
        r[4] = p[4];
    }
};

template <> struct VolLoad<DT_BF16> {
    typedef uint16_t T;
    static constexpr int kRowSlack = 1;
    static __device__ __forceinline__ float one(const uint16_t *p)
    {
        return __uint_as_float((uint32_t)(*p) << 16);
    }
    static __device__ __forceinline__ void row5(const uint16_t *p, float (&r)[5])
    {
        u3 a;
        __builtin_memcpy(&a, p, 12);
        r[0] = __uint_as_float(a.x << 16); r[1] = __uint_as_float(a.x & 0xffff0000u);
        r[2] = __uint_as_float(a.y << 16); r[3] = __uint_as_float(a.y & 0xffff0000u);
        r[4] = __uint_as_float(a.z << 16);
    }
};

template <> struct VolLoad<DT_F16> {
    typedef uint16_t T;
    static constexpr int kRowSlack = 1;
    static __device__ __forceinline__ float h2f(uint32_t bits)
    {
        __half_raw raw;
        raw.x = (unsigned short)(bits & 0xffffu);
        return __half2float(__half(raw));
    }
    static __device__ __forceinline__ float one(const uint16_t *p) { return h2f(*p); }
    static __device__ __forceinline__ void row5(const uint16_t *p, float (&r)[5])
    {
        u3 a;
        __builtin_memcpy(&a, p, 12);
        r[0] = h2f(a.x); r[1] = h2f(a.x >> 16);
        r[2] = h2f(a.y); r[3] = h2f(a.y >> 16);
        r[4] = h2f(a.z);
    }
};

// ---------------------------------------------------------------------------
// Forward projection (gpuForwardProject.cu:4-101).
// Work item = (direction, 16x16 pixel tile); one pixel per thread; wave = 16x4
// pixels.  The KB table sits in LDS.  For kerHWidth 2 the 5x5x5 gather is
// unrolled with one unaligned vector load per x-row; other widths use the
// generic loop.
// ---------------------------------------------------------------------------
// n / d for n < 2^31 by a multiplication (d and so the shift wave-uniform).
struct FastDiv {
    unsigned d, mul, shift;
    void set(unsigned div)
    {
        d = div;
        unsigned l = 0;
        while ((1ull << l) < div) l++;
        shift = l + 31;
        mul = (unsigned)(((1ull << shift) + div - 1) / div);
    }
    __device__ __forceinline__ unsigned operator()(unsigned n) const
    {
        return (unsigned)(((unsigned long long)n * mul) >> shift);
    }
};

// fp_lds_kernel's order of the 8x8 tiles.  A workgroup takes 2 x 2 tiles, the
// hardware deals workgroups round-robin to the 8 XCDs, and each XCD walks
// whole images (or, for few directions, whole bands of images) of its own, so
// that neighbouring tiles, whose voxel boxes overlap, share that XCD's L2.
// Walking the tiles row by row over all XCDs kept vertical neighbours on one
// XCD only where a row of workgroups is a multiple of 8 (N=64, 128, 256):
// 500 random directions 1,280 -> 828 us at N=160, 1,743 -> 1,205 at N=192,
// 2,048 at N=96 1,568 -> 1,208, 2,000 at N=128 2,183 -> 2,068.
struct FPWalk {
    FastDiv unitTiles;  // workgroup tiles of a unit (a band of one image)
    FastDiv cols;       // workgroup tiles across an image
    FastDiv bands;      // units per image
    unsigned rows, bandRows;  // workgroup tile rows of an image, of a band
    unsigned units, perXcd;   // units in all; workgroup tiles of one XCD's list
    unsigned turn;            // 7: the XCDs change places from 8 units to the next (bands), 0: not
};

struct FPArgs {
    const void *vol;
    const float *axes;
    float *out;
    const float *ker;
    int V, M, K, nAxes;
    float maskR, kerScale, kerCenter, fW;
    int convW, tilesPerRow, tilesPerImg;
    unsigned perXcd, totalWork;
    int maskD2;  // fp_lds_kernel: largest integer d2 with sqrtf((float)d2) <= maskR (-1: none)
    const unsigned *check;  // fp_lds_kernel with the 501-entry table: launch_check_volume's flag, or null
    FPWalk walk;            // fp_lds_kernel: its order of the tiles
    const unsigned *columns;  // adj_lds_kernel: launch_check_back's flag when the column launches came first, or null
    float orthTol;            // with columns: frames they took are orthonormal to this
};

constexpr int KFP_FAST = 501;  // the table the mixed-volume launch requires (kerScale 125, kerCenter 250)

template <int DT, bool W2>
__global__ __launch_bounds__(kThreads) void fp_kernel(FPArgs p)
{
    using L = VolLoad<DT>;
    using T = typename L::T;
    __shared__ float sker[kMaxKerSize];

    const unsigned work = xcd_work(p.perXcd);
    if (work >= p.totalWork) return;  // uniform per block
    for (int t = threadIdx.x; t < p.K; t += kThreads) sker[t] = p.ker[t];
    __syncthreads();

    const int a = (int)(work / (unsigned)p.tilesPerImg);
    const int tile = (int)(work - (unsigned)a * (unsigned)p.tilesPerImg);
    const int ty = tile / p.tilesPerRow, tx = tile - ty * p.tilesPerRow;
    const int i = tx * 16 + (threadIdx.x & 15), j = ty * 16 + (threadIdx.x >> 4);
    const int M = p.M, V = p.V;
    if (i >= M || j >= M) return;
    const int ci = M / 2, cv = V / 2;

    float r = sqrtf((float)(i - ci) * (i - ci) + (j - ci) * (j - ci));
    float acc = 0.f;
    if (r <= p.maskR) {
        const float *ax = p.axes + (size_t)9 * a;
        const float u0 = ax[0], u1 = ax[1], u2 = ax[2];
        const float v0 = ax[3], v1 = ax[4], v2 = ax[5];
        const float fi = (float)(i - ci), fj = (float)(j - ci);
        const float x = ref_sum2c(u0, fi, v0, fj, (float)cv);
        const float y = ref_sum2c(u1, fi, v1, fj, (float)cv);
        const float z = ref_sum2c(u2, fi, v2, fj, (float)cv);
        const int X = (int)roundf(x), Y = (int)roundf(y), Z = (int)roundf(z);
        const T *vol = (const T *)p.vol;
        const long long V3 = (long long)V * V * V;

        if (W2) {
            float wi[5], wj[5], wk[5];
#pragma unroll
            for (int t = 0; t < 5; t++) {
                wi[t] = sker[kb_index((float)(X - 2 + t) - x, p.fW, p.kerScale, p.kerCenter, p.K)];
                wj[t] = sker[kb_index((float)(Y - 2 + t) - y, p.fW, p.kerScale, p.kerCenter, p.K)];
                wk[t] = sker[kb_index((float)(Z - 2 + t) - z, p.fW, p.kerScale, p.kerCenter, p.K)];
            }
            float wij[5][5];
#pragma unroll
            for (int aa = 0; aa < 5; aa++)
#pragma unroll
                for (int bb = 0; bb < 5; bb++) wij[aa][bb] = wi[aa] * wj[bb];

            // unsigned: X may be INT_MAX (a non-finite direction)
            const unsigned top = (unsigned)max(V - 4, 0), topX = (unsigned)max(V - 4 - L::kRowSlack, 0);
            const bool fast = (unsigned)X - 2u < topX && (unsigned)Y - 2u < top && (unsigned)Z - 2u < top;
            if (fast) {
                const T *base = vol + (((size_t)(Z - 2) * V + (size_t)(Y - 2)) * V + (X - 2));
#pragma unroll
                for (int cc = 0; cc < 5; cc++) {
#pragma unroll
                    for (int bb = 0; bb < 5; bb++) {
                        float rv[5];
                        L::row5(base + ((size_t)cc * V + bb) * V, rv);
#pragma unroll
                        for (int aa = 0; aa < 5; aa++) acc = fmaf(wij[aa][bb] * wk[cc], rv[aa], acc);
                    }
                }
            } else {
                // Neighbourhood leaves the volume (only with a user mask radius
                // beyond the default or non-unit axes): the reference's
                // linear-index test (gpuForwardProject.cu:90), plus a lower
                // bound so nothing is read before the volume.
#pragma unroll
                for (int aa = 0; aa < 5; aa++)
#pragma unroll
                    for (int bb = 0; bb < 5; bb++)
#pragma unroll
                        for (int cc = 0; cc < 5; cc++) {
                            long long lin = ((long long)Z - 2 + cc) * V * V +
                                            ((long long)Y - 2 + bb) * V + ((long long)X - 2 + aa);
                            if (lin < V3 && lin >= 0)
                                acc = fmaf(wij[aa][bb] * wk[cc], L::one(vol + lin), acc);
                        }
            }
        } else {
            const int W = p.convW;
            for (int i1 = X - W; i1 <= X + W; i1++) {
                float wi = sker[kb_index((float)i1 - x, p.fW, p.kerScale, p.kerCenter, p.K)];
                for (int j1 = Y - W; j1 <= Y + W; j1++) {
                    float wj = sker[kb_index((float)j1 - y, p.fW, p.kerScale, p.kerCenter, p.K)];
                    for (int k1 = Z - W; k1 <= Z + W; k1++) {
                        float wk = sker[kb_index((float)k1 - z, p.fW, p.kerScale, p.kerCenter, p.K)];
                        float w = wi * wj * wk;
                        long long lin = (long long)k1 * V * V + (long long)j1 * V + i1;
                        if (lin < V3 && lin >= 0) acc = fmaf(w, L::one(vol + lin), acc);
                    }
                }
            }
        }
    }
    p.out[(size_t)a * M * M + (size_t)j * M + i] = acc;
}

// ---------------------------------------------------------------------------
// Forward projection, LDS-staged (kerHWidth 2).  A workgroup is 4 waves; each
// wave owns one 8x8 pixel tile of one direction.  The wave stages into LDS the
// axis-aligned box of volume voxels its pixels' 5x5x5 stencils can touch
// (bounded from the tile's four corner positions, about 30 voxels per pixel),
// reading each box row as unaligned 16-byte segments, and gathers the 125 taps
// from LDS instead of issuing 25 scattered row loads per pixel to the texture
// path.  A tile whose box exceeds the per-wave LDS budget is staged and
// gathered as two 8x4 halves, and a half whose box still does not fit gathers
// from global memory.  The gather is arranged as
// acc += wk[c] * sum_ab (wi[a]*wj[b]) * vol, i.e. the reference's product
// (wi*wj)*wk regrouped: rounding decisions are unchanged, only FP32
// accumulation rounding differs.
// ---------------------------------------------------------------------------
constexpr int FPT = 8;          // tile edge (pixels)
// Per-wave staged box budgets (floats): 5-wide windows and the transpose, and
// 4-wide windows, which leave room for the phase table.  Four boxes take at
// most 40,960 bytes of LDS, a quarter of the CU's 160 KB, so four workgroups
// share a CU (the kernel's VGPRs allow four waves per SIMD).  The median box
// of an 8x8 tile's 5-wide windows at N=128 holds 2,464 floats; nearly every
// box of the 4-wide ones fits.  Boxes that do not are staged as two 8x4
// halves.  Five workgroups per CU with 1,920 floats ran the 4-wide gather 10%
// slower.
constexpr int FPBOX = 2560;
constexpr int FPBOX4 = 2432;
constexpr int FPKER = 640;      // generic-table path: table floats kept in LDS

__device__ __forceinline__ void wave_lds_sync_fp()
{
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// floor(x + 0.5) in one instruction; equals roundf(x) for x >= 0.5 (below,
// an FP32 x + 0.5 can round up to the next integer).
__device__ __forceinline__ int cvt_rpi(float x)
{
    int i;
    asm("v_cvt_rpi_i32_f32 %0, %1" : "=v"(i) : "v"(x));
    return i;
}

// 501-entry table lookup (see bp_fast_kernel for the exactness argument) from
// the table in global memory (2 KB, cache-resident): 5-wide windows, and tiles
// of 4-wide ones that cannot take the phase table.  Clamping the index to [0,
// 500] picks the entry the reference's clamp of r would (|r| <= 2.5 here), and
// keeps any index, even from a non-finite coordinate, inside the table.
__device__ __forceinline__ float kb_fast_fp(const float *__restrict__ ker, float r)
{
    const float s = fmaf(r, 125.0f, 250.0f);
    const int i = cvt_rpi(s);
    return *(const float *)((const char *)ker + (unsigned)min(max(i, 0), 500) * 4u);
}

template <typename L>
__device__ __forceinline__ void load4(const typename L::T *p, float (&v)[4]);
template <>
__device__ __forceinline__ void load4<VolLoad<DT_F32>>(const float *p, float (&v)[4])
{
    f4 a;
    __builtin_memcpy(&a, p, 16);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
}
template <>
__device__ __forceinline__ void load4<VolLoad<DT_BF16>>(const uint16_t *p, float (&v)[4])
{
    typedef unsigned int u2 __attribute__((ext_vector_type(2)));
    u2 a;
    __builtin_memcpy(&a, p, 8);
    v[0] = __uint_as_float(a.x << 16); v[1] = __uint_as_float(a.x & 0xffff0000u);
    v[2] = __uint_as_float(a.y << 16); v[3] = __uint_as_float(a.y & 0xffff0000u);
}
template <>
__device__ __forceinline__ void load4<VolLoad<DT_F16>>(const uint16_t *p, float (&v)[4])
{
    typedef unsigned int u2 __attribute__((ext_vector_type(2)));
    u2 a;
    __builtin_memcpy(&a, p, 8);
    v[0] = VolLoad<DT_F16>::h2f(a.x); v[1] = VolLoad<DT_F16>::h2f(a.x >> 16);
    v[2] = VolLoad<DT_F16>::h2f(a.y); v[3] = VolLoad<DT_F16>::h2f(a.y >> 16);
}

// Tile body.  W4 = false: every pixel gathers its full 5x5x5 stencil from the
// box of all its stencils.  W4 = true (501-entry table whose end entries are 0,
// volume known to be finite): along each axis the reference's taps X-2..X+2
// (X = roundf(x)) have r = tap - x clamped to [-2, 2], and the tap with r <= -2
// reads table entry 0 and the one with r >= 2 entry 500 (fma(-2, 125, 250) = 0
// and fma(2, 125, 250) = 500 exactly).  If x >= X, then X - 2 - x <= -2; if
// x < X, then X + 2 - x > 2: one of the two end taps always has weight 0, and
// the others are the four taps from Xs = X - 2 + (x >= X) = floor(x) - 1.  The
// zero taps add fma(0, v, s) = s for finite v, so gathering the 4x4x4 window
// gives the same sums bit for bit, and the box shrinks to the voxels the
// windows touch: [floor(min) - 1, floor(max) + 2] per axis instead of
// [floor(min) - 2, ceil(max) + 2], about 40% fewer voxels to stage.
template <int DT, bool FAST, bool W4, bool BIG, int BOX>
__device__ __forceinline__ void fp_lds_tile_body(const FPArgs &p, const float *__restrict__ sker,
                                                 const f4 *__restrict__ phase, float *__restrict__ box, int a, int i0,
                                                 int j0, int ln, bool active, bool pix, float *out)
{
    using L = VolLoad<DT>;
    using T = typename L::T;
    constexpr int NW = W4 ? 4 : 5;  // taps per axis
    const int i = i0 + (ln & 7), j = j0 + (ln >> 3);
    const int M = p.M, V = p.V, ci = M / 2, cv = V / 2;
    const float *ax = p.axes + (size_t)9 * a;
    const float u0 = ax[0], u1 = ax[1], u2 = ax[2];
    const float v0 = ax[3], v1 = ax[4], v2 = ax[5];
    const float fi = (float)(i - ci), fj = (float)(j - ci);
    const float x = ref_sum2c(u0, fi, v0, fj, (float)cv);
    const float y = ref_sum2c(u1, fi, v1, fj, (float)cv);
    const float z = ref_sum2c(u2, fi, v2, fj, (float)cv);
    // centre and first tap of each axis' window
    int X = 0, Y = 0, Z = 0, Xs, Ys, Zs;
    if (W4) {
        Xs = (int)floorf(x) - 1; Ys = (int)floorf(y) - 1; Zs = (int)floorf(z) - 1;
    } else {
        X = (int)roundf(x); Y = (int)roundf(y); Z = (int)roundf(z);
        Xs = X - 2; Ys = Y - 2; Zs = Z - 2;
    }

    const long long V3 = (long long)V * V * V;
    const T *vol = (const T *)p.vol;

    float wi[NW], wj[NW], wk[NW];
    bool single = true;
    int least = NW;  // of a box's edges
    if constexpr (W4) {
        // The four entries of an axis' window lie 125 apart: one index, of the
        // last tap, and one row (T[k], T[k + 125], T[k + 250], T[k + 375]) of
        // the phase table.  The first taps' indices are that one's minus
        // multiples of 125 unless its FP32 value is exactly a half-integer
        // (see ColVisit's argument) or the position below 1, where tap - x may
        // be rounded; then every lane looks its taps up one by one.  One row
        // read (5 ns per wave and CU) replaces four table gathers through the
        // texture path (10 ns each); with the four-dword rows below 2,196 ->
        // 1,997 us per 2,000 directions at N=128.
        if (phase != nullptr) {
            const float sx = fmaf((float)(Xs + 3) - x, 125.0f, 250.0f);
            const float sy = fmaf((float)(Ys + 3) - y, 125.0f, 250.0f);
            const float sz = fmaf((float)(Zs + 3) - z, 125.0f, 250.0f);
            const auto half = [](float s) {  // or NaN
                const float f = __builtin_amdgcn_fractf(s);
                return !(f < 0.5f || f > 0.5f);
            };
            const bool odd = half(sx) || half(sy) || half(sz) || !(fminf(x, fminf(y, z)) >= 1.0f);
            single = __ballot(active && odd) != 0ull;
            // a coordinate of NaN or beyond all volumes gets the row of zeros,
            // as its lookups tap by tap read entries 0 and 500
            const f4 qx = phase[min(max(cvt_rpi(sx), 374), 500) - 374];
            const f4 qy = phase[min(max(cvt_rpi(sy), 374), 500) - 374];
            const f4 qz = phase[min(max(cvt_rpi(sz), 374), 500) - 374];
#pragma unroll
            for (int t = 0; t < NW; t++) {
                wi[t] = qx[t];
                wj[t] = qy[t];
                wk[t] = qz[t];
            }
        }
    }
    if (single) {
        // A direction with an infinite component has pixels at 0 times infinity
        // whose windows lie outside the box that the corners give: no box then.
        if (__ballot(active && !(x + y + z == x + y + z)) != 0ull) least = INT_MAX;
#pragma unroll
        for (int t = 0; t < NW; t++) {
            if (FAST) {
                wi[t] = kb_fast_fp(p.ker, (float)(Xs + t) - x);
                wj[t] = kb_fast_fp(p.ker, (float)(Ys + t) - y);
                wk[t] = kb_fast_fp(p.ker, (float)(Zs + t) - z);
            } else {
                wi[t] = sker[kb_index((float)(Xs + t) - x, p.fW, p.kerScale, p.kerCenter, p.K)];
                wj[t] = sker[kb_index((float)(Ys + t) - y, p.fW, p.kerScale, p.kerCenter, p.K)];
                wk[t] = sker[kb_index((float)(Zs + t) - z, p.fW, p.kerScale, p.kerCenter, p.K)];
            }
        }
    }

    // Stages the voxel box of pixel rows j0 + rlo .. j0 + rhi of the tile and
    // gathers the pixels of the lanes with mine set; false (nothing done) when
    // the box does not fit the wave's LDS budget.  Uniform across the wave.
    float acc = 0.f;
    auto stageAndGather = [&](int rlo, int rhi, bool mine, auto splitT) -> bool {
        // Box from the corners: positions are affine in (i, j), so every
        // pixel's coordinate lies in [min corner, max corner] (the 1e-3 margin
        // covers FP32 evaluation error), widened by the window.
        const float ai = (float)(i0 - ci), bi = (float)(i0 + FPT - 1 - ci);
        const float aj = (float)(j0 + rlo - ci), bj = (float)(j0 + rhi - ci);
        auto lo = [&](float uu, float vv) {
            return (int)floorf(fminf(uu * ai, uu * bi) + fminf(vv * aj, vv * bj) + (float)cv - 1e-3f) - (W4 ? 1 : 2);
        };
        auto hi = [&](float uu, float vv) {
            const float e = fmaxf(uu * ai, uu * bi) + fmaxf(vv * aj, vv * bj) + (float)cv + 1e-3f;
            return (int)(W4 ? floorf(e) : ceilf(e)) + 2;
        };
        const int bx0 = __builtin_amdgcn_readfirstlane(lo(u0, v0));
        const int by0 = __builtin_amdgcn_readfirstlane(lo(u1, v1));
        const int bz0 = __builtin_amdgcn_readfirstlane(lo(u2, v2));
        const int Dx = __builtin_amdgcn_readfirstlane(hi(u0, v0)) - bx0 + 1;
        const int Dy = __builtin_amdgcn_readfirstlane(hi(u1, v1)) - by0 + 1;
        const int Dz = __builtin_amdgcn_readfirstlane(hi(u2, v2)) - bz0 + 1;
        // Volume addressing by 32-bit byte offsets: from the volume's base
        // (below 4 GB), or (BIG) from the box's first element, whose
        // linear-index span is below 64 V^2 elements.
        if (!(Dx >= least && Dy >= NW && Dz >= NW && Dx <= 64 && Dy <= 64 && Dz <= 64 &&
              (BIG ? 64LL * V * V : V3) * (long long)sizeof(T) < (1LL << 32)))
            return false;
        // 16-byte segments per box row; for the 5-wide windows enough that the
        // 8-wide read (below) stays inside the row's staged segments.
        const int segs = W4 ? (Dx + 3) >> 2 : (Dx + 8 - NW) >> 2;
        // LDS pitches (floats), multiples of 4 (16-byte rows).  When the box
        // still fits, the row and plane pitches are padded to an odd number
        // of 16-byte units so that the rows and planes a tile's pixels read
        // spread over the banks (a pitch of 16 puts every row at the same
        // bank offset); otherwise the rows are packed.
        int RP = (segs | 1) * 4;
        int PP = RP * Dy + ((Dy & 1) ? 0 : RP);
        if (PP * Dz > BOX) {
            RP = segs * 4;
            PP = RP * Dy;
        }
        if (PP * Dz > BOX) return false;

        // Stage.  A plane of the box holds P = Dy * segs row segments.  With
        // P <= 64 one pass covers G = 64 / P planes (lane -> plane offset pl,
        // row ey, segment sg), else G = 1 and a plane takes ceil(P / 64) lane
        // passes; each lane then steps through its planes with one add for
        // the volume offset and one for the LDS pointer.  The lane -> task
        // divisions use the reciprocal: (q + 0.5) / P is at least 0.5 / P
        // away from an integer, far more than its error for q, P <= 1024.
        const int VV = V * V;
        const int P = Dy * segs;
        const float rP = __builtin_amdgcn_rcpf((float)P), rSegs = __builtin_amdgcn_rcpf((float)segs);
        const int G = P <= 64 ? __builtin_amdgcn_readfirstlane((int)(64.5f * rP)) : 1;
        const int nLanePass = (P + 63) >> 6;
        // The reference bounds only the linear index (gpuForwardProject.cu:90):
        // when the box's whole index range is inside the volume no element
        // needs a check.  lin grows with ez, ey and the segment, so the range
        // is spanned by the first and last segment of the box.
        const long long linLo = (long long)bz0 * VV + (long long)by0 * V + bx0;
        const long long linHi = linLo + (long long)(Dz - 1) * VV + (long long)(Dy - 1) * V + 4 * segs - 1;
        const bool boxIn = linLo >= 0 && linHi < V3;
        // Four planes per batch (three with the 16-bit types' conversions; six
        // for 5-wide windows): all loads of a batch are in flight before the
        // first LDS store waits on them (2, 3, 4, 5 and 6 planes: 2.17, 2.10,
        // 2.07, 2.08 and 2.08 ms per 2,000 directions at N=128; BF16, 500 at
        // N=256: 2.49, 2.28, -, 2.45 and 2.48 ms; 8 needs more than 128 VGPRs,
        // three waves per SIMD).  The checked and unchecked variants are separate loops
        // (boxIn is wave-uniform).  The unchecked one addresses the volume by
        // a 32-bit byte offset from the volume's base, or (BIG: volumes of
        // 4 GB and more) from the box's first element; the checked one, which
        // runs only on boxes that cross the volume's index range, by the
        // linear index in 32 or (BIG) 64 bits, unsigned: it wraps for boxes
        // at infinity, and as a signed one could pass the test in 32 bits and
        // be an address in 64.
        const T *volBox = vol + ((BIG && boxIn) ? linLo : 0);
        using Lin = std::conditional_t<BIG, unsigned long long, unsigned>;
        constexpr int SB = DT != DT_F32 ? 3 : W4 ? 4 : 6;
        const int lStep = G * VV, dStep = G * PP;
        for (int c = 0; c < nLanePass; c++) {
            const int q = ln + 64 * c;
            const int pl = (int)(((float)q + 0.5f) * rP);
            const int pq = q - pl * P;
            const int ey = (int)(((float)pq + 0.5f) * rSegs);
            const int sg = pq - ey * segs;
            if (pl >= G) continue;
            const Lin lin0 = ((Lin)bz0 + (Lin)pl) * (Lin)VV + ((Lin)by0 + (Lin)ey) * (Lin)V + ((Lin)bx0 + (Lin)(4 * sg));
            float *d0 = box + pl * PP + ey * RP + 4 * sg;
            auto stage = [&](auto inBox) {
                // offset from volBox (BIG and boxIn: inside the box's span,
                // below 2^30) or the linear index
                using Idx = std::conditional_t<decltype(inBox)::value, int, Lin>;
                Idx l = (Idx)((BIG && decltype(inBox)::value) ? lin0 - (Lin)linLo : lin0);
                float *dp = d0;
                for (int ez = pl; ez < Dz; ez += SB * G) {
                    float v4[SB][4];
#pragma unroll
                    for (int k = 0; k < SB; k++) {
                        if (ez + k * G < Dz) {
                            const Idx lk = l + (Idx)(k * lStep);
                            if (decltype(inBox)::value) {
                                load4<L>((const T *)((const char *)volBox + (unsigned)lk * (unsigned)sizeof(T)), v4[k]);
                            } else {
#pragma unroll
                                for (int e = 0; e < 4; e++) {
                                    const Lin le = (Lin)lk + (Lin)e;
                                    v4[k][e] = le < (Lin)V3 ? L::one(vol + le) : 0.f;
                                }
                            }
                        }
                    }
#pragma unroll
                    for (int k = 0; k < SB; k++) {
                        if (ez + k * G < Dz) {
                            f4 w4 = {v4[k][0], v4[k][1], v4[k][2], v4[k][3]};
                            *(f4 *)(dp + k * dStep) = w4;
                        }
                    }
                    l += (Idx)(SB * lStep);
                    dp += SB * dStep;
                }
            };
            if (boxIn) {
                stage(std::true_type{});
            } else {
                stage(std::false_type{});
            }
        }
        // 4-wide windows: a row is four dwords (two paired reads, no
        // alignment), 64 products instead of the 128 of aligned 16-byte units.
        auto planeSum4 = [&](const float *bq, const float (&wx)[NW], const float (&wy)[NW], int cc) {
            float sc = 0.f;
#pragma unroll
            for (int bb = 0; bb < NW; bb++) {
                float v[4];
                __builtin_memcpy(v, bq + cc * PP + bb * RP, 16);
                float row = wx[0] * v[0];
#pragma unroll
                for (int aa = 1; aa < 4; aa++) row = fmaf(wx[aa], v[aa], row);
                sc = fmaf(wy[bb], row, sc);
            }
            return sc;
        };
        // 5-wide windows: each 5-tap row is read as the two aligned 16-byte
        // units that contain it, [xo - o, xo - o + 8) with o = xo & 3, and the
        // x weights are shifted by o with zeros in the unused slots.  Since
        // xo <= Dx - NW, xo - o + 8 <= 4 * floor((Dx - NW) / 4) + 8, which
        // is at most 4 * segs, so the read stays inside the row's staged
        // segments.  The unused values are staged volume values times 0,
        // which leaves every sum bit-identical to the NW-tap read when they
        // are finite.  With the 5-wide window a non-finite one makes the
        // pixel's sum NaN (0 * NaN and 0 * Inf are NaN), so a pixel whose sum
        // is not finite is gathered again with the 5-tap read, and NaN and Inf
        // reach exactly the pixels whose stencil holds them, as in the
        // reference; the 4-wide window runs only on finite volumes.
        wave_lds_sync_fp();
        // x weights shifted by o (zeros in the unused slots) times the y weights.
        auto shifted = [&](const float (&wx)[NW], const float (&wy)[NW], int o, float (&w8)[8][NW]) {
            float ws[8];
#pragma unroll
            for (int t = 0; t < 8; t++) {
                float w = 0.f;
#pragma unroll
                for (int sft = 0; sft < 4; sft++)
                    if (t - sft >= 0 && t - sft < NW) w = (o == sft) ? wx[t - sft] : w;
                ws[t] = w;
            }
#pragma unroll
            for (int t = 0; t < 8; t++)
#pragma unroll
                for (int bb = 0; bb < NW; bb++) w8[t][bb] = ws[t] * wy[bb];
        };
        // One z plane of a window: NW rows of the 16-byte read.
        auto planeSum = [&](const float *bq, const float (&w8)[8][NW], int cc) {
            float sc = 0.f;
#pragma unroll
            for (int bb = 0; bb < NW; bb++) {
                const float *rp = bq + cc * PP + bb * RP;
                const f4 q0 = *(const f4 *)rp, q1 = *(const f4 *)(rp + 4);
                sc = fmaf(w8[0][bb], q0.x, sc);
                sc = fmaf(w8[1][bb], q0.y, sc);
                sc = fmaf(w8[2][bb], q0.z, sc);
                sc = fmaf(w8[3][bb], q0.w, sc);
                sc = fmaf(w8[4][bb], q1.x, sc);
                sc = fmaf(w8[5][bb], q1.y, sc);
                sc = fmaf(w8[6][bb], q1.z, sc);
                sc = fmaf(w8[7][bb], q1.w, sc);
            }
            return sc;
        };
        float res = 0.f;
        bool gathered = false;
        if constexpr (!decltype(splitT)::value) {
            if (active && mine) {
                const int xo = Xs - bx0, o = W4 ? 0 : xo & 3;
                const float *bq = box + (Zs - bz0) * PP + (Ys - by0) * RP + (xo - o);
                if constexpr (W4) {
#pragma unroll
                    for (int cc = 0; cc < NW; cc++) res = fmaf(wk[cc], planeSum4(bq, wi, wj, cc), res);
                } else {
                    float w8[8][NW];
                    shifted(wi, wj, o, w8);
#pragma unroll
                    for (int cc = 0; cc < NW; cc++) res = fmaf(wk[cc], planeSum(bq, w8, cc), res);
                }
                gathered = true;
            }
        } else {
            // Half tile: the lanes of the other half (lane ^ 32; their own
            // pixels are not in this box) gather the last two planes of their
            // partner's window while the owner gathers the first NW - 2, so
            // the wave reads 3 * NW rows per pixel instead of NW * NW; the
            // owner adds the parts.
            constexpr int H = NW - 2;  // planes the owner gathers
            const int pX = __shfl_xor(Xs, 32), pY = __shfl_xor(Ys, 32), pZ = __shfl_xor(Zs, 32);
            const int pAct = __shfl_xor(active ? 1 : 0, 32);
            float gwi[NW], gwj[NW];
#pragma unroll
            for (int t = 0; t < NW; t++) {
                const float a5 = __shfl_xor(wi[t], 32), b5 = __shfl_xor(wj[t], 32);
                gwi[t] = mine ? wi[t] : a5;
                gwj[t] = mine ? wj[t] : b5;
            }
            const float pkA = __shfl_xor(wk[H], 32), pkB = __shfl_xor(wk[H + 1], 32);
            const int gX = mine ? Xs : pX, gY = mine ? Ys : pY, gZ = mine ? Zs : pZ + H;
            const float k0 = mine ? wk[0] : pkA, k1 = mine ? wk[1] : pkB;
            float part = 0.f;
            if (mine ? active : pAct != 0) {
                const int xo = gX - bx0, o = W4 ? 0 : xo & 3;
                const float *bq = box + (gZ - bz0) * PP + (gY - by0) * RP + (xo - o);
                if constexpr (W4) {
                    part = fmaf(k0, planeSum4(bq, gwi, gwj, 0), part);
                    part = fmaf(k1, planeSum4(bq, gwi, gwj, 1), part);
                } else {
                    float w8[8][NW];
                    shifted(gwi, gwj, o, w8);
                    part = fmaf(k0, planeSum(bq, w8, 0), part);
                    part = fmaf(k1, planeSum(bq, w8, 1), part);
                    if (mine) part = fmaf(wk[2], planeSum(bq, w8, 2), part);
                }
            }
            const float other = __shfl_xor(part, 32);
            res = part + other;
            gathered = active && mine;
        }
        if (gathered) {
            if (!W4 && !__builtin_isfinite(res)) {
                const float *bp = box + (Z - 2 - bz0) * PP + (Y - 2 - by0) * RP + (X - 2 - bx0);
                res = 0.f;
#pragma unroll
                for (int cc = 0; cc < NW; cc++) {
                    float sc = 0.f;
#pragma unroll
                    for (int bb = 0; bb < NW; bb++) {
                        const float *rp = bp + cc * PP + bb * RP;
#pragma unroll
                        for (int aa = 0; aa < NW; aa++) sc = fmaf(wi[aa] * wj[bb], rp[aa], sc);
                    }
                    res = fmaf(wk[cc], sc, res);
                }
            }
            acc = res;
        }
        wave_lds_sync_fp();  // the box is read before it is staged again
        return true;
    };

    // The whole 8x8 tile; if its box is too large, its two 8x4 halves one
    // after the other; a half that still does not fit gathers from global
    // memory.
    bool done = stageAndGather(0, FPT - 1, true, std::false_type{});
    if (!done) {
        const bool top = (ln >> 3) < FPT / 2;
        const bool d0 = stageAndGather(0, FPT / 2 - 1, top, std::true_type{});
        const bool d1 = stageAndGather(FPT / 2, FPT - 1, !top, std::true_type{});
        done = top ? d0 : d1;
    }
    if (!done && active) {
#pragma unroll
        for (int cc = 0; cc < NW; cc++) {
            float sc = 0.f;
#pragma unroll
            for (int bb = 0; bb < NW; bb++)
#pragma unroll
                for (int aa = 0; aa < NW; aa++) {
                    const long long lin = ((long long)Zs + cc) * V * V + ((long long)Ys + bb) * V + ((long long)Xs + aa);
                    if (lin < V3 && lin >= 0) sc = fmaf(wi[aa] * wj[bb], L::one(vol + lin), sc);
                }
            acc = fmaf(wk[cc], sc, acc);
        }
    }
    if (pix) *out = active ? acc : 0.f;
}

// One 8x8 tile of one direction; W4 (only with the 501-entry table) selects
// the 4-wide windows.
template <int DT, bool FAST, bool W4, bool BIG, int BOX>
__device__ __forceinline__ void fp_lds_tile(const FPArgs &p, const float *__restrict__ sker,
                                            const f4 *__restrict__ phase, float *__restrict__ box, int a, int tx, int ty,
                                            int ln)
{
    const int i0 = tx * FPT, j0 = ty * FPT;
    const int i = i0 + (ln & 7), j = j0 + (ln >> 3);
    const int M = p.M, ci = M / 2;
    const bool pix = i < M && j < M;

    // sqrtf(d2) <= maskR for the exact integer d2, as one integer compare
    // (sqrtf is monotone; the host finds the largest passing d2).
    const bool active = pix && (i - ci) * (i - ci) + (j - ci) * (j - ci) <= p.maskD2;
    float *out = p.out + (size_t)a * M * M + (size_t)j * M + i;
    if (__ballot(active) == 0ull) {
        if (pix) *out = 0.f;
        return;
    }
    fp_lds_tile_body<DT, FAST, FAST && W4, BIG, BOX>(p, sker, phase, box, a, i0, j0, ln, active, pix, out);
}

// The 4-wide windows need a finite volume and a finite 501-entry table whose
// end entries are 0 (the reference's table sets them so): launch_check_volume
// writes *check = 1 when they hold.  Wave-uniform.
__device__ __forceinline__ bool fp_win4(const unsigned *check)
{
    return check != nullptr && __builtin_amdgcn_readfirstlane(*check) == 1u;
}

// A row of zeros, then (T[k], T[k + 125], T[k + 250], T[k + 375]), k <= 125, of
// the 501-entry table, by the whole workgroup.
constexpr int FPPHASE = 127;
__device__ __forceinline__ void fp_phase_table(f4 *__restrict__ phase, const float *__restrict__ ker)
{
    for (int k = threadIdx.x; k < FPPHASE; k += kThreads) {
        const float *t = ker + max(k - 1, 0);
        const f4 row = {t[0], t[125], t[250], t[375]};
        phase[k] = k > 0 ? row : f4{0.f, 0.f, 0.f, 0.f};
    }
    __syncthreads();
}

template <int DT, bool FAST, bool BIG>
__global__ __launch_bounds__(kThreads) void fp_lds_kernel(FPArgs p)
{
    __shared__ float sker[FPKER];
    // four boxes of 5-wide windows, or four boxes of 4-wide ones and the phase table
    __shared__ __attribute__((aligned(16))) float sbox[4 * FPBOX];
    static_assert(4 * FPPHASE + 4 * FPBOX4 <= 4 * FPBOX, "the phase table and its boxes");
    f4 *const sphase = (f4 *)(sbox + 4 * FPBOX4);

    if (!FAST) {  // the fast lookup reads the table from global memory
        for (int t = threadIdx.x; t < p.K; t += kThreads) sker[t] = p.ker[t];
        __syncthreads();
    }
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), ln = threadIdx.x & 63;
    const FPWalk &wk = p.walk;
    const unsigned xcd = blockIdx.x & 7u;
    auto walk = [&](auto win4) {
        for (unsigned it = blockIdx.x >> 3; it < wk.perXcd; it += gridDim.x >> 3) {
            const unsigned k = wk.unitTiles(it), t = it - k * wk.unitTiles.d;
            const unsigned unit = ((xcd + (k & wk.turn)) & 7u) + 8u * k;
            const unsigned a = wk.bands(unit), band = unit - a * wk.bands.d;
            const unsigned r = wk.cols(t), row = band * wk.bandRows + r, col = t - r * wk.cols.d;
            const int tx = (int)(2u * col) + (wv & 1), ty = (int)(2u * row) + (wv >> 1);
            if (unit >= wk.units || row >= wk.rows || tx >= p.tilesPerRow || ty >= p.tilesPerRow) continue;
            constexpr bool W4 = decltype(win4)::value;
            constexpr int BOX = W4 ? FPBOX4 : FPBOX;
            fp_lds_tile<DT, FAST, W4, BIG, BOX>(p, sker, W4 ? sphase : nullptr, sbox + wv * BOX,
                                                (int)a, tx, ty, ln);
        }
    };
    // The window width is chosen once, outside the tile loop, so that each
    // loop is register-allocated on its own.
    if (FAST && fp_win4(p.check)) {
        fp_phase_table(sphase, p.ker);
        walk(std::true_type{});
    } else {
        walk(std::false_type{});
    }
}

// ---------------------------------------------------------------------------
// Exact transpose of the forward gather: each in-mask pixel scatters its
// value through the same (voxel, weight) pairs with FP32 atomics.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kThreads) void adj_kernel(FPArgs p, const float *__restrict__ img,
                                                       float *__restrict__ volAcc)
{
    __shared__ float sker[kMaxKerSize];
    const unsigned work = xcd_work(p.perXcd);
    if (work >= p.totalWork) return;
    for (int t = threadIdx.x; t < p.K; t += kThreads) sker[t] = p.ker[t];
    __syncthreads();

    const int a = (int)(work / (unsigned)p.tilesPerImg);
    const int tile = (int)(work - (unsigned)a * (unsigned)p.tilesPerImg);
    const int ty = tile / p.tilesPerRow, tx = tile - ty * p.tilesPerRow;
    const int i = tx * 16 + (threadIdx.x & 15), j = ty * 16 + (threadIdx.x >> 4);
    const int M = p.M, V = p.V;
    if (i >= M || j >= M) return;
    const int ci = M / 2, cv = V / 2;
    float r = sqrtf((float)(i - ci) * (i - ci) + (j - ci) * (j - ci));
    if (!(r <= p.maskR)) return;
    const float val = img[(size_t)a * M * M + (size_t)j * M + i];
    if (val == 0.f) return;
    const float *ax = p.axes + (size_t)9 * a;
    const float u0 = ax[0], u1 = ax[1], u2 = ax[2];
    const float v0 = ax[3], v1 = ax[4], v2 = ax[5];
    const float fi = (float)(i - ci), fj = (float)(j - ci);
    const float x = ref_sum2c(u0, fi, v0, fj, (float)cv);
    const float y = ref_sum2c(u1, fi, v1, fj, (float)cv);
    const float z = ref_sum2c(u2, fi, v2, fj, (float)cv);
    const int X = (int)roundf(x), Y = (int)roundf(y), Z = (int)roundf(z);
    const long long V3 = (long long)V * V * V;
    const int W = p.convW;
    for (int i1 = X - W; i1 <= X + W; i1++) {
        float wi = sker[kb_index((float)i1 - x, p.fW, p.kerScale, p.kerCenter, p.K)];
        for (int j1 = Y - W; j1 <= Y + W; j1++) {
            float wj = sker[kb_index((float)j1 - y, p.fW, p.kerScale, p.kerCenter, p.K)];
            for (int k1 = Z - W; k1 <= Z + W; k1++) {
                float wk = sker[kb_index((float)k1 - z, p.fW, p.kerScale, p.kerCenter, p.K)];
                float w = wi * wj * wk;
                long long lin = (long long)k1 * V * V + (long long)j1 * V + i1;
                if (lin < V3 && lin >= 0 && w != 0.f) unsafeAtomicAdd(volAcc + lin, w * val);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Forward projection over several volumes in one launch (the request
// server's batches mix volumes of different N).  Each segment is a run of
// directions on one volume with its own geometry and output; work items are
// the segments' 8x8 tiles, numbered segment after segment, and every wave
// finds its segment by a binary search over the segments' first work items
// (wave-uniform, so the search and the descriptor reads are scalar).  The
// tile code is fp_lds_tile's, so each image is bit-identical to a launch of
// its own volume alone.  A batch of requests on several volumes is one launch;
// its workgroups walk the work list three tiles per wave.
// ---------------------------------------------------------------------------
template <int DT, bool BIG>
__global__ __launch_bounds__(kThreads) void fp_lds_multi_kernel(FPMultiArgs m)
{
    __shared__ __attribute__((aligned(16))) float sbox[4][FPBOX4];
    __shared__ f4 sphase[FPPHASE];
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), ln = threadIdx.x & 63;
    fp_phase_table(sphase, m.seg[0].ker);  // segments with another table look up tap by tap
    for (unsigned work = blockIdx.x * 4u + (unsigned)wv; work < m.totalWork; work += gridDim.x * 4u) {
        int lo = 0, hi = m.nSegs - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (m.seg[mid].workStart <= work) lo = mid; else hi = mid - 1;
        }
        const FPSegment &sg = m.seg[lo];
        FPArgs a;
        a.vol = sg.vol; a.axes = sg.axes; a.out = sg.out; a.ker = sg.ker;
        a.V = sg.V; a.M = sg.M; a.K = KFP_FAST; a.nAxes = sg.nAxes;
        a.maskR = 0.f; a.kerScale = 125.0f; a.kerCenter = 250.0f; a.fW = 2.0f;
        a.convW = 2; a.tilesPerRow = sg.tilesPerRow; a.tilesPerImg = sg.tilesPerImg;
        a.perXcd = 0; a.totalWork = 0; a.maskD2 = sg.maskD2; a.check = sg.check;
        a.columns = nullptr; a.orthTol = 0.f;
        const f4 *phase = sg.ker == m.seg[0].ker ? sphase : nullptr;
        const unsigned local = work - sg.workStart;
        const int d = (int)(local / (unsigned)sg.tilesPerImg), tile = (int)(local - (unsigned)d * (unsigned)sg.tilesPerImg);
        const int ty = tile / sg.tilesPerRow, tx = tile - ty * sg.tilesPerRow;
        if (fp_win4(sg.check)) fp_lds_tile<DT, true, true, BIG, FPBOX4>(a, nullptr, phase, sbox[wv], d, tx, ty, ln);
        else fp_lds_tile<DT, true, false, BIG, FPBOX4>(a, nullptr, nullptr, sbox[wv], d, tx, ty, ln);
    }
}

// The transpose has no use for a direction's third vector: a9[6..8] = u x v,
// true when [u v] is orthonormal to tol.
__device__ __forceinline__ bool adj_plane(float (&a)[9], float tol)
{
    a[6] = a[1] * a[5] - a[2] * a[4];
    a[7] = a[2] * a[3] - a[0] * a[5];
    a[8] = a[0] * a[4] - a[1] * a[3];
    return fabsf(a[0] * a[0] + a[1] * a[1] + a[2] * a[2] - 1.f) <= tol &&
           fabsf(a[3] * a[3] + a[4] * a[4] + a[5] * a[5] - 1.f) <= tol &&
           fabsf(a[0] * a[3] + a[1] * a[4] + a[2] * a[5]) <= tol;
}

// ---------------------------------------------------------------------------
// Exact transpose, LDS-box scatter (kerHWidth 2, tables of at most FPKER
// entries).  A wave owns one 8x8 pixel tile of one direction, as in
// fp_lds_tile: it bounds the voxel box its pixels' 5x5x5 stencils touch (the
// same corner bound), zeroes that box in LDS, adds every tap's w * value into
// it (ordered plain read-modify-write in rounds that keep colliding lanes
// apart; LDS float atomics for frames that are not orthonormal), and adds each touched
// box voxel to the volume with one global atomic: about 11 global atomics per
// pixel at N=128 instead of one per tap (125).  Box voxels map to the volume through the reference's
// linear index (gpuForwardProject.cu:90), so the transpose keeps the forward
// gather's row wrap.  A tile whose box exceeds the LDS budget runs as two 8x4
// halves; a half that still does not fit scatters with global atomics.  With
// launch_check_volume's flag over the CAS images and the table (all finite,
// table ends 0) it scatters only the 4x4x4 windows of the taps that can have
// nonzero weight, from the windows' smaller box, as fp_lds_tile_body gathers
// them: the skipped taps add w * value = 0.
// ---------------------------------------------------------------------------
template <bool FAST, bool W4>
__device__ __forceinline__ void adj_lds_tile(const FPArgs &p, const float *__restrict__ sker,
                                             float *__restrict__ box, const float *__restrict__ img,
                                             float *__restrict__ volAcc, unsigned work, int ln, bool skewOnly)
{
    const int a = (int)(work / (unsigned)p.tilesPerImg);
    const int tile = (int)(work - (unsigned)a * (unsigned)p.tilesPerImg);
    const int ty = tile / p.tilesPerRow, tx = tile - ty * p.tilesPerRow;
    const int i0 = tx * FPT, j0 = ty * FPT;
    const int i = i0 + (ln & 7), j = j0 + (ln >> 3);
    const int M = p.M, V = p.V, ci = M / 2, cv = V / 2;
    const bool pix = i < M && j < M;
    const bool inMask = pix && (i - ci) * (i - ci) + (j - ci) * (j - ci) <= p.maskD2;
    const float val = inMask ? img[(size_t)a * M * M + (size_t)j * M + i] : 0.f;
    const bool act = inMask && val != 0.f;
    if (__ballot(act) == 0ull) return;

    const float *ax = p.axes + (size_t)9 * a;
    const float u0 = ax[0], u1 = ax[1], u2 = ax[2];
    const float v0 = ax[3], v1 = ax[4], v2 = ax[5];
    if (skewOnly) {  // the column launches have done the orthonormal planes
        float f[9] = {u0, u1, u2, v0, v1, v2, 0.f, 0.f, 0.f};
        if (adj_plane(f, p.orthTol)) return;
    }
    const float fi = (float)(i - ci), fj = (float)(j - ci);
    const float x = ref_sum2c(u0, fi, v0, fj, (float)cv);
    const float y = ref_sum2c(u1, fi, v1, fj, (float)cv);
    const float z = ref_sum2c(u2, fi, v2, fj, (float)cv);
    const int X = (int)roundf(x), Y = (int)roundf(y), Z = (int)roundf(z);
    // Window of each axis: all five taps, or (W4, checked images and table)
    // the four that can have nonzero weight, from floor(x) - 1 (as in
    // fp_lds_tile_body).
    constexpr int NW = W4 ? 4 : 5;
    const int Xs = X - 2 + ((W4 && x >= (float)X) ? 1 : 0);
    const int Ys = Y - 2 + ((W4 && y >= (float)Y) ? 1 : 0);
    const int Zs = Z - 2 + ((W4 && z >= (float)Z) ? 1 : 0);
    const long long V3 = (long long)V * V * V;
    const long long VV = (long long)V * V;
    // [u v] orthonormal to 1e-4 (wave-uniform: one direction per tile)
    const bool orthoFrame = fabsf(u0 * u0 + u1 * u1 + u2 * u2 - 1.f) <= 1e-4f &&
                            fabsf(v0 * v0 + v1 * v1 + v2 * v2 - 1.f) <= 1e-4f &&
                            fabsf(u0 * v0 + u1 * v1 + u2 * v2) <= 1e-4f;

    float wi[NW], wj[NW], wk[NW];
#pragma unroll
    for (int t = 0; t < NW; t++) {
        if (FAST) {
            wi[t] = kb_fast_fp(p.ker, (float)(Xs + t) - x);
            wj[t] = kb_fast_fp(p.ker, (float)(Ys + t) - y);
            wk[t] = kb_fast_fp(p.ker, (float)(Zs + t) - z);
        } else {
            wi[t] = sker[kb_index((float)(Xs + t) - x, p.fW, p.kerScale, p.kerCenter, p.K)];
            wj[t] = sker[kb_index((float)(Ys + t) - y, p.fW, p.kerScale, p.kerCenter, p.K)];
            wk[t] = sker[kb_index((float)(Zs + t) - z, p.fW, p.kerScale, p.kerCenter, p.K)];
        }
    }

    // The reference's bounds test on the linear index, one global atomic per
    // tap (gpuForwardProject.cu:90); every tap of the window, as the box path.
    auto scatterGlobal = [&]() {
#pragma unroll
        for (int cc = 0; cc < NW; cc++)
#pragma unroll
            for (int bb = 0; bb < NW; bb++)
#pragma unroll
                for (int aa = 0; aa < NW; aa++) {
                    const long long lin = (long long)(Zs + cc) * VV + (long long)(Ys + bb) * V + (Xs + aa);
                    const float w = wi[aa] * wj[bb] * wk[cc];
                    if (lin < V3 && lin >= 0) unsafeAtomicAdd(volAcc + lin, w * val);
                }
    };

    // Scatters the pixels of the tile rows j0 + rlo .. j0 + rhi (lanes with
    // mine set) through an LDS box; false (nothing done) when the box does not
    // fit the wave's budget.  Uniform across the wave.
    auto scatter = [&](int rlo, int rhi, bool mine) -> bool {
        const float ai = (float)(i0 - ci), bi = (float)(i0 + FPT - 1 - ci);
        const float aj = (float)(j0 + rlo - ci), bj = (float)(j0 + rhi - ci);
        auto lo = [&](float uu, float vv) {
            return (int)floorf(fminf(uu * ai, uu * bi) + fminf(vv * aj, vv * bj) + (float)cv - 1e-3f) - (W4 ? 1 : 2);
        };
        auto hi = [&](float uu, float vv) {
            const float e = fmaxf(uu * ai, uu * bi) + fmaxf(vv * aj, vv * bj) + (float)cv + 1e-3f;
            return (int)(W4 ? floorf(e) : ceilf(e)) + 2;
        };
        const int bx0 = __builtin_amdgcn_readfirstlane(lo(u0, v0));
        const int by0 = __builtin_amdgcn_readfirstlane(lo(u1, v1));
        const int bz0 = __builtin_amdgcn_readfirstlane(lo(u2, v2));
        const int Dx = __builtin_amdgcn_readfirstlane(hi(u0, v0)) - bx0 + 1;
        const int Dy = __builtin_amdgcn_readfirstlane(hi(u1, v1)) - by0 + 1;
        const int Dz = __builtin_amdgcn_readfirstlane(hi(u2, v2)) - bz0 + 1;
        if (!(Dx >= NW && Dy >= NW && Dz >= NW && Dx <= 64 && Dy <= 64 && Dz <= 64)) return false;
        const int RP = Dx, PP = Dx * Dy, total = PP * Dz;
        if (total > FPBOX) return false;
        for (int e = ln; e < total; e += 64) box[e] = 0.f;
        wave_lds_sync_fp();
        // Every finite in-row pixel's stencil lies inside the box (the corner
        // bound); a lane whose does not (non-finite directions) scatters
        // through the checked global path instead of outside its box.
        const bool inBox = (unsigned)(Xs - bx0) <= (unsigned)(Dx - NW) &&
                           (unsigned)(Ys - by0) <= (unsigned)(Dy - NW) &&
                           (unsigned)(Zs - bz0) <= (unsigned)(Dz - NW);
        if (act && mine && !inBox) scatterGlobal();
        const int key = (Zs - bz0) * PP + (Ys - by0) * RP + (Xs - bx0);
        // Tap value (wi * val) * (wj * wk): the forward weight times the pixel
        // value, grouped so that only NW + NW * NW products are live across
        // the rounds instead of one per tap (the per-tap products, hoisted
        // out of the rounds loop, held the kernel at 225 VGPRs).
        float wiv[NW];
#pragma unroll
        for (int aa = 0; aa < NW; aa++) wiv[aa] = wi[aa] * val;
        auto addStencil = [&](bool atomic) {
            float *bq = box + key;
#pragma unroll 1
            for (int cc = 0; cc < NW; cc++)
#pragma unroll
                for (int bb = 0; bb < NW; bb++) {
                    float *rp = bq + cc * PP + bb * RP;
                    const float wjk = wj[bb] * wk[cc];
#pragma unroll
                    for (int aa = 0; aa < NW; aa++) {
                        const float t = wiv[aa] * wjk;
                        if (atomic) {
                            atomicAdd(rp + aa, t);
                        } else {
                            rp[aa] = rp[aa] + t;
                            // Keep this tap's write before the next tap's read:
                            // another lane's stencil may cover this word at a
                            // later tap, and its read must see this write.
                            __asm__ volatile("" ::: "memory");
                        }
                    }
                }
        };
        bool pend = act && mine && inBox;
        if (orthoFrame) {
            // Plain read-modify-write, one tap after the other (LDS float
            // atomics ran 3.6x slower: 40 vs 11 ms at N=96 with 2,048
            // directions).  One wave's LDS instructions execute in order and
            // each tap's read follows the previous tap's write (compiler
            // barrier), so a lane's read sees every earlier write of every
            // lane; only lanes of the same instruction can lose an update,
            // and those target the same word at every tap exactly when their
            // windows start at the same voxel (key).  The start is X - 2 with
            // X = roundf(x), or floor(x) - 1 with the 4-wide windows, per axis;
            // for an orthonormal frame two pixels whose starts coincide have
            // positions less than 1 apart in every coordinate, so they are at
            // most sqrt(3) apart: tile neighbours.  A lane waits while a lower
            // pending neighbour (left, up, up-left, up-right) has its key;
            // every round serves at least the lowest pending lane of each key.
            const int ix = ln & 7, jy = ln >> 3;
            while (__ballot(pend) != 0ull) {
                const int k = pend ? key : -1 - ln;  // distinct for lanes not pending
                const int kl = __shfl(k, ln - 1), ku = __shfl(k, ln - 8);
                const int kul = __shfl(k, ln - 9), kur = __shfl(k, ln - 7);
                const bool wait = pend && ((ix >= 1 && kl == k) || (jy >= 1 && ku == k) ||
                                           (ix >= 1 && jy >= 1 && kul == k) || (ix <= 6 && jy >= 1 && kur == k));
                if (pend && !wait) addStencil(false);
                pend = wait;
                wave_lds_sync_fp();
            }
        } else if (pend) {
            addStencil(true);
        }
        wave_lds_sync_fp();
        // Flush the touched voxels plane by plane; a lane takes elements
        // q = ln, ln + 64, ... of a plane (row ey = q / RP by the reciprocal,
        // exact for q, RP <= 4096).
        const float rRP = __builtin_amdgcn_rcpf((float)RP);
        for (int ez = 0; ez < Dz; ez++) {
            const float *bp = box + ez * PP;
            const long long zbase = (long long)(bz0 + ez) * VV + (long long)by0 * V + bx0;
            for (int q = ln; q < PP; q += 64) {
                const float s = bp[q];
                if (s != 0.f) {
                    const int ey = (int)(((float)q + 0.5f) * rRP);
                    const int ex = q - ey * RP;
                    const long long lin = zbase + (long long)ey * V + ex;
                    if (lin >= 0 && lin < V3) unsafeAtomicAdd(volAcc + lin, s);
                }
            }
        }
        wave_lds_sync_fp();  // the box is read before it is zeroed again
        return true;
    };

    bool done = scatter(0, FPT - 1, true);
    if (!done) {
        const bool top = (ln >> 3) < FPT / 2;
        const bool d0 = scatter(0, FPT / 2 - 1, top);
        const bool d1 = scatter(FPT / 2, FPT - 1, !top);
        done = top ? d0 : d1;
    }
    if (!done && act) scatterGlobal();
}

template <bool FAST>
__global__ __launch_bounds__(kThreads) void adj_lds_kernel(FPArgs p, const float *__restrict__ img,
                                                           float *__restrict__ volAcc)
{
    __shared__ float sker[FPKER];
    __shared__ float sbox[4][FPBOX];
    // What the column launches have left (launch_check_back's flag): all
    // frames, those that are not orthonormal, or none.
    const unsigned done = p.columns != nullptr ? (unsigned)__builtin_amdgcn_readfirstlane(*p.columns) : 0u;
    if (done == 3u) return;
    if (!FAST) {
        for (int t = threadIdx.x; t < p.K; t += kThreads) sker[t] = p.ker[t];
        __syncthreads();
    }
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), ln = threadIdx.x & 63;
    if (FAST && (done != 0u || fp_win4(p.check))) {
        for (unsigned work = blockIdx.x * 4u + (unsigned)wv; work < p.totalWork; work += gridDim.x * 4u)
            adj_lds_tile<FAST, true>(p, sker, sbox[wv], img, volAcc, work, ln, done != 0u);
    } else {
        for (unsigned work = blockIdx.x * 4u + (unsigned)wv; work < p.totalWork; work += gridDim.x * 4u)
            adj_lds_tile<FAST, false>(p, sker, sbox[wv], img, volAcc, work, ln, false);
    }
}

// ---------------------------------------------------------------------------
// Back projection, reference semantics (gpuBackProject.cu:4-113), as an
// owner-computes gather: a workgroup owns an 8x8x4 voxel brick, culls the
// directions whose slab |n.(v-c)| <= kerHWidth cannot touch the brick, keeps
// the survivors in LDS in direction order, and each thread accumulates its own
// voxel.  No atomics: launches on one volume must be stream-ordered.
// ---------------------------------------------------------------------------
struct BPArgs {
    float *vol;
    float *dens;
    const float *axes;
    const float *img;
    const float *ker;
    int V, M, K, nAxes;
    float maskR, kerScale, kerCenter, fW, hw;
    int convW, bricksX, bricksXY;
    int maskD2;  // largest integer d2 with sqrtf((float)d2) <= maskR (-1: none)
    int posRound;  // bp_fast_kernel: in-mask voxels of orthonormal frames project to fi, fj >= 0.5
    int maskLo;    // smallest coordinate of an in-mask voxel (V/2 - floor(sqrt(maskD2)))
    const int *order;  // bp_fast_kernel, col_kernel: brick (block) id per work item, heaviest first
    unsigned perXcd, totalWork;
    const unsigned *check;  // bp_fast_kernel: launch_check_back's flag, or null
    float orthTol;          // frames that the column launches take are orthonormal to this
};

constexpr int BPX = 8, BPY = 8, BPZ = 4;

template <bool DENS>
__global__ __launch_bounds__(kThreads) void bp_kernel(BPArgs p)
{
    __shared__ float sker[kMaxKerSize];
    __shared__ float sax[kThreads * 9];
    __shared__ int sidx[kThreads];
    __shared__ int swave[kThreads / 64];

    const unsigned work = xcd_work(p.perXcd);
    if (work >= p.totalWork) return;
    const int bz = (int)(work / (unsigned)p.bricksXY);
    const int rem = (int)(work - (unsigned)bz * (unsigned)p.bricksXY);
    const int by = rem / p.bricksX, bx = rem - by * p.bricksX;
    const int ox = bx * BPX, oy = by * BPY, oz = bz * BPZ;
    const int V = p.V, M = p.M, cv = V / 2, ci = M / 2;

    // Whole brick outside the mask sphere: nothing to do (uniform exit).
    {
        float dx = fmaxf(fmaxf((float)(ox - cv), (float)(cv - (ox + BPX - 1))), 0.f);
        float dy = fmaxf(fmaxf((float)(oy - cv), (float)(cv - (oy + BPY - 1))), 0.f);
        float dz = fmaxf(fmaxf((float)(oz - cv), (float)(cv - (oz + BPZ - 1))), 0.f);
        if (dx * dx + dy * dy + dz * dz > (p.maskR + 1.f) * (p.maskR + 1.f)) return;
    }
    const int t = threadIdx.x;
    for (int k = t; k < p.K; k += kThreads) sker[k] = p.ker[k];

    const int vi = ox + (t & 7), vj = oy + ((t >> 3) & 7), vk = oz + (t >> 6);
    const bool inVol = vi < V && vj < V && vk < V;
    const float rr = sqrtf((float)(vi - cv) * (vi - cv) + (vj - cv) * (vj - cv) + (vk - cv) * (vk - cv));
    const bool active = inVol && (rr <= p.maskR);
    const float dvi = (float)vi - cv, dvj = (float)vj - cv, dvk = (float)vk - cv;
    const float fvi = (float)vi, fvj = (float)vj, fvk = (float)vk, cvf = (float)cv;
    const float bcx = (float)ox + 0.5f * (BPX - 1) - (float)cv;
    const float bcy = (float)oy + 0.5f * (BPY - 1) - (float)cv;
    const float bcz = (float)oz + 0.5f * (BPZ - 1) - (float)cv;
    const int M2 = M * M;

    double accAll = 0.0, densAll = 0.0;
    const int wv = t >> 6, ln = t & 63;

    for (int base = 0; base < p.nAxes; base += kThreads) {
        const int n = min(kThreads, p.nAxes - base);
        __syncthreads();  // previous list consumed (and table loaded)
        bool pass = false;
        float a9[9];
        if (t < n) {
            const float *ax = p.axes + (size_t)9 * (base + t);
#pragma unroll
            for (int k = 0; k < 9; k++) a9[k] = ax[k];
            const float d = bcx * a9[6] + bcy * a9[7] + bcz * a9[8];
            const float sup = 0.5f * (BPX - 1) * fabsf(a9[6]) + 0.5f * (BPY - 1) * fabsf(a9[7]) +
                              0.5f * (BPZ - 1) * fabsf(a9[8]);
            pass = fabsf(d) <= p.hw + sup + 1e-3f;
        }
        const unsigned long long bal = __ballot(pass);
        if (ln == 0) swave[wv] = __popcll(bal);
        __syncthreads();
        int off = 0, total = 0;
#pragma unroll
        for (int w = 0; w < kThreads / 64; w++) {
            off += (w < wv) ? swave[w] : 0;
            total += swave[w];
        }
        if (pass) {
            const int pos = off + __popcll(bal & ((1ull << ln) - 1ull));
            sidx[pos] = base + t;
#pragma unroll
            for (int k = 0; k < 9; k++) sax[pos * 9 + k] = a9[k];
        }
        __syncthreads();

        for (int q = 0; q < total; q++) {
            const float *ax = sax + q * 9;
            const float n0 = ax[6], n1 = ax[7], n2 = ax[8];
            const float fk = ref_sum3(dvi, n0, dvj, n1, dvk, n2);
            if (!(active && fabsf(fk) <= p.hw)) continue;
            const float u0 = ax[0], u1 = ax[1], u2 = ax[2];
            const float v0 = ax[3], v1 = ax[4], v2 = ax[5];
            const float fi = ref_sum3(dvi, u0, dvj, u1, dvk, u2) + (float)ci;
            const float fj = ref_sum3(dvi, v0, dvj, v1, dvk, v2) + (float)ci;
            const int I = (int)roundf(fi), J = (int)roundf(fj);
            const float *im = p.img + (size_t)sidx[q] * M2;
            float cum = 0.f, dsum = 0.f;
            if (p.convW == 2) {
                // Tap position fl(fma(di, u, fl(dj*v)) + c): the products
                // dj*v are rounded once per row, di stays exact.
                float Di[5], Bx[5], By[5], Bz[5];
#pragma unroll
                for (int s = 0; s < 5; s++) {
                    const float dj = (float)(J - 2 + s - ci);
                    Di[s] = (float)(I - 2 + s - ci);
                    Bx[s] = dj * v0; By[s] = dj * v1; Bz[s] = dj * v2;
                }
#pragma unroll
                for (int jj = 0; jj < 5; jj++) {
#pragma unroll
                    for (int ii = 0; ii < 5; ii++) {
                        const float px = fmaf(Di[ii], u0, Bx[jj]) + cvf;
                        float w = sker[kb_index(px - fvi, p.fW, p.kerScale, p.kerCenter, p.K)];
                        const float py = fmaf(Di[ii], u1, By[jj]) + cvf;
                        w = w * sker[kb_index(py - fvj, p.fW, p.kerScale, p.kerCenter, p.K)];
                        const float pz = fmaf(Di[ii], u2, Bz[jj]) + cvf;
                        w = w * sker[kb_index(pz - fvk, p.fW, p.kerScale, p.kerCenter, p.K)];
                        const unsigned lin = ((unsigned)J - 2u + jj) * (unsigned)M + ((unsigned)I - 2u + ii);
                        if (lin < (unsigned)M2) {
                            cum = cum + im[lin] * w;
                            if (DENS) dsum = dsum + w;
                        }
                    }
                }
            } else {
                const int W = p.convW;
                for (int j1 = J - W; j1 <= J + W; j1++) {
                    for (int i1 = I - W; i1 <= I + W; i1++) {
                        const float ti = (float)(i1 - ci), tj = (float)(j1 - ci);
                        const float px = ref_sum2c(ti, u0, tj, v0, cvf);
                        float w = sker[kb_index(px - fvi, p.fW, p.kerScale, p.kerCenter, p.K)];
                        const float py = ref_sum2c(ti, u1, tj, v1, cvf);
                        w = w * sker[kb_index(py - fvj, p.fW, p.kerScale, p.kerCenter, p.K)];
                        const float pz = ref_sum2c(ti, u2, tj, v2, cvf);
                        w = w * sker[kb_index(pz - fvk, p.fW, p.kerScale, p.kerCenter, p.K)];
                        const unsigned lin = (unsigned)j1 * (unsigned)M + (unsigned)i1;
                        if (lin < (unsigned)M2) {
                            cum = cum + im[lin] * w;
                            if (DENS) dsum = dsum + w;
                        }
                    }
                }
            }
            accAll += (double)cum;
            if (DENS) densAll += (double)dsum;
        }
    }
    if (active) {
        const size_t vidx = ((size_t)vk * V + vj) * V + vi;
        p.vol[vidx] = (float)((double)p.vol[vidx] + accAll);
        if (DENS) p.dens[vidx] = (float)((double)p.dens[vidx] + densAll);
    }
}

// ---------------------------------------------------------------------------
// Back projection fast path (kerHWidth 2, 501-entry table: kerScale 125,
// kerCenter 250), same reference semantics as bp_kernel.
//
// Work layout.  A workgroup owns an 8x8x8 brick and the list of directions
// whose slab can touch it (culled and compacted in direction order, as in
// bp_kernel).  Wave w takes list entries w, w+4, w+8, ...  For each direction
// the wave first finds the brick voxels inside the slab |fk| <= 2 (lane l
// tests the 8 voxels of column (l & 7, l >> 3)), compacts them into a
// per-wave queue in LDS, and then runs the 25-tap gather on 64 queued voxels
// at a time, so every lane carries an active voxel (a fixed voxel-per-lane
// layout leaves most lanes idle: a slab activates ~1/3 of a brick).
// The queue spans directions (entries carry a 7-bit direction slot), so the
// tail of one direction fills up with the next and groups stay full.  Two
// entries of one group can name the same voxel (different directions), so
// contributions go to a per-wave LDS accumulator one direction after the
// other (plain read-modify-writes: a float LDS atomic holds the LDS for 194
// cycles per wave, against 8; 7.58 -> 6.92 ms per 2,000 directions at N=128,
// 2.67 -> 2.29 ms with the density, 777 at N=64); the waves' accumulators
// are combined in a fixed order at the end and added to the volume in FP64.
//
// Table index.  The reference, as contracted, takes
// k = roundf(fma(clamp(r, -2, 2), 125, 250)) with r = fl(p - v).  For every
// FP32 r in [-4.5, 4.5], floor(fma(r, 125, 250) + 0.5) saturated to [0, 500]
// equals k (checked exhaustively, with floor(s + 0.5) exact and with s + 0.5
// first rounded to FP32, so the result does not depend on how the instruction
// rounds inside), and v_cvt_rpi_i32_f32 computes floor(x + 0.5) in one
// instruction.  The LDS table is padded on both sides with copies of its end
// entries, so offsets beyond +-2 land on the entry the reference's clamp
// would pick and r needs no clamp.
//
// Mask.  sqrtf(d2) <= maskRadius with d2 a small integer is monotone in d2,
// so the host passes the largest passing d2 and the test is an integer
// compare.
// ---------------------------------------------------------------------------
constexpr int BB = 8;                  // brick edge
constexpr int BV = BB * BB * BB;       // voxels per brick
constexpr int KPAD = 320;              // padding entries on each side of the table
constexpr int KFAST = 501;
constexpr int KTOT = KFAST + 2 * KPAD; // padded table length
constexpr int QCAP = 1024;             // per-wave queue ring (>= BV + 64, power of 2)
constexpr int BPCH = 128;              // directions culled per pass (queue entries hold 9-bit voxel + 7-bit slot)

__device__ __forceinline__ float kb_fast(const float *__restrict__ sk, float r)
{
    int i = cvt_rpi(fmaf(r, 125.0f, 250.0f));  // floor(s + 0.5)
    i = min(max(i, -KPAD), KFAST - 1 + KPAD);
    return sk[KPAD + i];
}

// Same lookup without the clamp, for directions whose frame is orthonormal
// (checked per chunk): then every tap has |r| <= 4.13 and the index stays in
// [-267, 767], inside the padding.
__device__ __forceinline__ float kb_fast_nc(const float *__restrict__ sk, float r)
{
    return sk[KPAD + cvt_rpi(fmaf(r, 125.0f, 250.0f))];
}

// Fused form of the same unclamped lookup for a tap at position p and an
// integer voxel coordinate v >= 3: where the reference's clamp is inactive
// (|p - v| <= 2) p >= 1, so p and v are multiples of ulp(p) and p - v is
// exact; then fma(r, 125, 250) = RN(125 p + 250 - 125 v) = fma(p, 125, c) with
// c = 250 - 125 v an exact integer.  Where |p - v| > 2 both sides saturate at
// table entry 0 or 500.  Checked for every float p in [v - 4.5, v + 4.5] and
// v in 3..4 and 9..2,100 (0 mismatches); v = 0, 1, 2 have mismatches.
constexpr int BP_FORM_A_MIN = 3;

__device__ __forceinline__ float kb_form(const float *__restrict__ sk, float pos, float c)
{
    return sk[KPAD + cvt_rpi(fmaf(pos, 125.0f, c))];
}

__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// [u v n] orthonormal to tol (false for non-finite frames).
__device__ __forceinline__ bool bp_orthonormal(const float (&a)[9], float tol)
{
    const float uu = a[0] * a[0] + a[1] * a[1] + a[2] * a[2];
    const float vv = a[3] * a[3] + a[4] * a[4] + a[5] * a[5];
    const float nn = a[6] * a[6] + a[7] * a[7] + a[8] * a[8];
    const float uv = a[0] * a[3] + a[1] * a[4] + a[2] * a[5];
    const float un = a[0] * a[6] + a[1] * a[7] + a[2] * a[8];
    const float vn = a[3] * a[6] + a[4] * a[7] + a[5] * a[8];
    return fabsf(uu - 1.f) <= tol && fabsf(vv - 1.f) <= tol && fabsf(nn - 1.f) <= tol &&
           fabsf(uv) <= tol && fabsf(un) <= tol && fabsf(vn) <= tol;
}

template <bool DENS, int BFW>
__global__ __launch_bounds__(64 * BFW) void bp_fast_kernel(BPArgs p)
{
    __shared__ float sker[KTOT];
    __shared__ float sax[BPCH * 9];
    __shared__ int sidx[BPCH];
    __shared__ int swave[BFW];
    __shared__ int snon[BFW];
    __shared__ float sacc[BFW][BV];
    __shared__ float sden[DENS ? BFW : 1][DENS ? BV : 1];
    __shared__ unsigned short squeue[BFW][QCAP];

    // Bricks near the centre meet every direction and bricks near the mask edge
    // few, so the order table puts the heavy (central) bricks first and
    // consecutive work items go round-robin to the XCDs.
    if (blockIdx.x >= p.totalWork) return;
    const unsigned work = (unsigned)p.order[blockIdx.x];
    const int bz = (int)(work / (unsigned)p.bricksXY);
    const int rem = (int)(work - (unsigned)bz * (unsigned)p.bricksXY);
    const int by = rem / p.bricksX, bx = rem - by * p.bricksX;
    const int ox = bx * BB, oy = by * BB, oz = bz * BB;
    const int V = p.V, M = p.M, cv = V / 2, ci = M / 2;
    {
        float dx = fmaxf(fmaxf((float)(ox - cv), (float)(cv - (ox + BB - 1))), 0.f);
        float dy = fmaxf(fmaxf((float)(oy - cv), (float)(cv - (oy + BB - 1))), 0.f);
        float dz = fmaxf(fmaxf((float)(oz - cv), (float)(cv - (oz + BB - 1))), 0.f);
        if (dx * dx + dy * dy + dz * dz > (p.maskR + 1.f) * (p.maskR + 1.f)) return;
    }
    // What the column launches have left: everything, the frames that are not
    // orthonormal, or nothing.
    const unsigned done = p.check != nullptr ? (unsigned)__builtin_amdgcn_readfirstlane(*p.check) : 0u;
    if (done == 3u) return;
    const int t = threadIdx.x;
    for (int k = t; k < KTOT; k += (64 * BFW)) sker[k] = p.ker[min(max(k - KPAD, 0), KFAST - 1)];
    for (int k = t; k < BFW * BV; k += (64 * BFW)) {
        (&sacc[0][0])[k] = 0.f;
        if (DENS) (&sden[0][0])[k] = 0.f;
    }

    // Orthonormal chunks use the fused lookup (kb_form) when every active
    // voxel of the brick has coordinates >= BP_FORM_A_MIN: the brick's corner
    // does, or the mask keeps every in-mask voxel there.
    const bool brickA = p.posRound &&
                        (min(ox, min(oy, oz)) >= BP_FORM_A_MIN || p.maskLo >= BP_FORM_A_MIN);

    const float cvf = (float)cv, cif = (float)ci;
    const float bc = 0.5f * (BB - 1);
    const float bcx = (float)ox + bc - cvf, bcy = (float)oy + bc - cvf, bcz = (float)oz + bc - cvf;
    const int M2 = M * M;
    const int wv = t >> 6, ln = t & 63;
    // This lane's voxel column for the slab test: (ox + cx, oy + cy, oz + 0..7).
    const int cx = ln & 7, cy = ln >> 3;
    const int vi0 = ox + cx, vj0 = oy + cy;
    unsigned vmask = 0;  // inside the volume and the mask sphere (direction-independent)
#pragma unroll
    for (int k = 0; k < BB; k++) {
        const int vk = oz + k;
        const int d2 = (vi0 - cv) * (vi0 - cv) + (vj0 - cv) * (vj0 - cv) + (vk - cv) * (vk - cv);
        if (vi0 < V && vj0 < V && vk < V && d2 <= p.maskD2) vmask |= 1u << k;
    }
    const float dvi0 = (float)vi0 - cv, dvj0 = (float)vj0 - cv;

    for (int base = 0; base < p.nAxes; base += BPCH) {
        const int n = min(BPCH, p.nAxes - base);
        __syncthreads();
        bool pass = false, orth = true;
        float a9[9];
        if (t < n) {
            const float *ax = p.axes + (size_t)9 * (base + t);
#pragma unroll
            for (int k = 0; k < 9; k++) a9[k] = ax[k];
            const float d = bcx * a9[6] + bcy * a9[7] + bcz * a9[8];
            const float sup = bc * (fabsf(a9[6]) + fabsf(a9[7]) + fabsf(a9[8]));
            pass = fabsf(d) <= p.hw + sup + 1e-3f;
            // rotation matrices are orthonormal to ~1e-7
            orth = bp_orthonormal(a9, 1e-4f);
            if (done != 0u && bp_orthonormal(a9, p.orthTol)) pass = false;
        }
        const unsigned long long bal = __ballot(pass);
        const unsigned long long nonOrth = __ballot(!orth);
        if (ln == 0) {
            swave[wv] = __popcll(bal);
            snon[wv] = nonOrth != 0ull;
        }
        __syncthreads();
        int non = 0;
#pragma unroll
        for (int w = 0; w < BFW; w++) non |= snon[w];
        const bool chunkOrtho = non == 0;
        int off = 0, total = 0;
#pragma unroll
        for (int w = 0; w < BFW; w++) {
            off += (w < wv) ? swave[w] : 0;
            total += swave[w];
        }
        if (pass) {
            const int pos = off + __popcll(bal & ((1ull << ln) - 1ull));
            sidx[pos] = base + t;
#pragma unroll
            for (int k = 0; k < 9; k++) sax[pos * 9 + k] = a9[k];
        }
        __syncthreads();

        // Directions of this chunk that wave wv handles: q = wv, wv + BFW, ...
        // Their active voxels stream through the wave's FIFO queue; every
        // full group of 64 entries is gathered with all lanes busy.
        int head = 0, tail = 0;  // queue indices (uniform), ring of size QCAP
        for (int q = wv; q < total || tail > head; q += BFW) {
            if (q < total) {
                const float *ax = sax + q * 9;
                const float n0 = ax[6], n1 = ax[7], n2 = ax[8];
                // Slab test of the lane's column (the reference's contracted
                // fk = fma(dvk, n2, fma(dvi, n0, fl(dvj * n1)))), appended to
                // the queue in (z, lane) order.
                const float fk0 = fmaf(dvi0, n0, dvj0 * n1);
#pragma unroll
                for (int k = 0; k < BB; k++) {
                    const float dvk = (float)(oz + k) - cv;
                    const float fk = fmaf(dvk, n2, fk0);
                    const bool on = ((vmask >> k) & 1u) && fabsf(fk) <= p.hw;
                    const unsigned long long b = __ballot(on);
                    if (on)
                        squeue[wv][(tail + __popcll(b & ((1ull << ln) - 1ull))) & (QCAP - 1)] =
                            (unsigned short)((cx + BB * (cy + BB * k)) | (q << 9));
                    tail += __popcll(b);
                }
            }
            const bool last = q + BFW >= total;
            wave_lds_sync();
            // Gather full groups (and, after the last direction, the rest).
            auto gather = [&](auto formT) {
            while (tail - head >= 64 || (last && tail > head)) {
                const int e = head + ln;
                head = min(head + 64, tail);
                if (e < tail) {
                    const unsigned ent = squeue[wv][e & (QCAP - 1)];
                    const int vox = ent & 511, qq = ent >> 9;
                    const float *ax = sax + qq * 9;
                    const float u0 = ax[0], u1 = ax[1], u2 = ax[2];
                    const float v0 = ax[3], v1 = ax[4], v2 = ax[5];
                    const float *im = p.img + (size_t)sidx[qq] * M2;
                    const int lx = vox & 7, ly = (vox >> 3) & 7, lz = vox >> 6;
                    const int vi = ox + lx, vj = oy + ly, vk = oz + lz;
                    const float dvi = (float)vi - cv, dvj = (float)vj - cv, dvk = (float)vk - cv;
                    const float fi = ref_sum3(dvi, u0, dvj, u1, dvk, u2) + cif;
                    const float fj = ref_sum3(dvi, v0, dvj, v1, dvk, v2) + cif;
                    constexpr int KF = decltype(formT)::value;
                    // The fused variant runs only when posRound holds (fi, fj >= 0.5),
                    // where floor(x + 0.5) is roundf(x) and one instruction.
                    const int I = KF > 0 ? cvt_rpi(fi) : (int)roundf(fi);
                    const int J = KF > 0 ? cvt_rpi(fj) : (int)roundf(fj);
                    const float fvi = (float)vi, fvj = (float)vj, fvk = (float)vk;
                    // Form constants 250 - 125 v (exact; used by the fused variant).
                    const float cX = fmaf(-125.0f, fvi, 250.0f);
                    const float cY = fmaf(-125.0f, fvj, 250.0f);
                    const float cZ = fmaf(-125.0f, fvk, 250.0f);
                    float Di[5];
#pragma unroll
                    for (int s5 = 0; s5 < 5; s5++) Di[s5] = (float)(I - 2 + s5 - ci);
                    float cum = 0.f, dsum = 0.f;
                    // unsigned, as the linear index below: I and J may be INT_MAX (a
                    // non-finite direction), where a signed sum could pass the test
                    // wrapped and be an address unwrapped
                    const unsigned top = (unsigned)max(M - 4, 0);
                    const bool inside = (unsigned)I - 2u < top && (unsigned)J - 2u < top;
#pragma unroll 1
                    for (int jj = 0; jj < 5; jj++) {
                        const float dj = (float)(J - 2 + jj - ci);
                        const float Bx = dj * v0, By = dj * v1, Bz = dj * v2;
                        float val[5], vin[5];  // image values; 1 where the tap is in bounds, else 0
                        const unsigned row = ((unsigned)J - 2u + jj) * (unsigned)M + ((unsigned)I - 2u);
                        if (inside) {
                            f4 a;
                            __builtin_memcpy(&a, im + row, 16);
                            val[0] = a.x; val[1] = a.y; val[2] = a.z; val[3] = a.w;
                            val[4] = im[row + 4];
#pragma unroll
                            for (int ii = 0; ii < 5; ii++) vin[ii] = 1.f;
                        } else {
                            // Reference bound on the linear index only
                            // (gpuBackProject.cu:99): wraps across rows.
#pragma unroll
                            for (int ii = 0; ii < 5; ii++) {
                                const unsigned lin = row + ii;
                                const bool ok = lin < (unsigned)M2;
                                val[ii] = ok ? im[lin] : 0.f;
                                vin[ii] = ok ? 1.f : 0.f;
                            }
                        }
#pragma unroll
                        for (int ii = 0; ii < 5; ii++) {
                            // fl(fma(di, u, fl(dj*v)) + c), the reference's contracted
                            // tap position (gpuBackProject.cu:77,84,91).
                            const float px = fmaf(Di[ii], u0, Bx) + cvf;
                            const float py = fmaf(Di[ii], u1, By) + cvf;
                            const float pz = fmaf(Di[ii], u2, Bz) + cvf;
                            float w, wy, wz;
                            if constexpr (KF < 0) {
                                w = kb_fast(sker, px - fvi);
                                wy = kb_fast(sker, py - fvj);
                                wz = kb_fast(sker, pz - fvk);
                            } else if constexpr (KF == 0) {
                                w = kb_fast_nc(sker, px - fvi);
                                wy = kb_fast_nc(sker, py - fvj);
                                wz = kb_fast_nc(sker, pz - fvk);
                            } else {
                                w = kb_form(sker, px, cX);
                                wy = kb_form(sker, py, cY);
                                wz = kb_form(sker, pz, cZ);
                            }
                            w = w * wy;
                            w = w * wz;
                            cum = fmaf(val[ii], w, cum);
                            // the density: the back projection of all-ones images
                            // (fma(1, w, d) = d + w, fma(0, w, d) = d)
                            if (DENS) dsum = fmaf(vin[ii], w, dsum);
                        }
                    }
                    // Two queued entries of one group can name the same voxel,
                    // but only for different directions: the adds go one
                    // direction after the other, as plain read-modify-writes
                    // (most groups hold one or two directions).  A wave's LDS
                    // instructions execute in order.
                    for (unsigned long long pend = __ballot(true); pend != 0ull;) {
                        const int first = __builtin_amdgcn_readlane(qq, __builtin_ctzll(pend));
                        const bool mine = qq == first;
                        if (mine) {
                            sacc[wv][vox] += cum;
                            if (DENS) sden[wv][vox] += dsum;
                        }
                        pend &= ~__ballot(mine);
                        __asm__ volatile("" ::: "memory");
                    }
                }
            }
            };
            if (!chunkOrtho) {
                gather(std::integral_constant<int, -1>{});
            } else if (brickA) {
                gather(std::integral_constant<int, 1>{});
            } else {
                gather(std::integral_constant<int, 0>{});
            }
            wave_lds_sync();  // queue slots consumed before they are refilled
            if (last) break;
        }
    }
    __syncthreads();
    for (int k = t; k < BV; k += (64 * BFW)) {
        const int lx = k & 7, ly = (k >> 3) & 7, lz = k >> 6;
        const int vi = ox + lx, vj = oy + ly, vk = oz + lz;
        if (vi >= V || vj >= V || vk >= V) continue;
        const int d2 = (vi - cv) * (vi - cv) + (vj - cv) * (vj - cv) + (vk - cv) * (vk - cv);
        if (d2 > p.maskD2) continue;
        const size_t vidx = ((size_t)vk * V + vj) * V + vi;
        double s = (double)p.vol[vidx];
#pragma unroll
        for (int w = 0; w < BFW; w++) s += (double)sacc[w][k];
        p.vol[vidx] = (float)s;
        if (DENS) {
            double d = (double)p.dens[vidx];
#pragma unroll
            for (int w = 0; w < BFW; w++) d += (double)sden[w][k];
            p.dens[vidx] = (float)d;
        }
    }
}

// ---------------------------------------------------------------------------
// Back projection, and the forward gather's exact transpose, by voxel columns:
// the path of orthonormal frames whose CAS images are finite (launch_check_back's
// flag; bp_fast_kernel or adj_lds_kernel runs what is left).
//
// bp_fast_kernel looks up three table entries for each of the 25 pixels of
// each voxel.  But a pixel's position does not depend on the voxel, and along
// the axis c on which the direction's normal is largest the plane's slab holds
// 4 to 7 consecutive voxels of a column.  So a lane owns a column and visits
// each pixel that can reach any of these voxels once: one position, one lookup
// for each of the two cross axes (shared by the column), and one index for all
// voxels of the column, whose entries lie 125 apart: the LDS table holds pairs
// (T[k], T[k - 125]), zero outside the table, and entry pairs 250 apart give
// the K weights in (K + 1) / 2 reads (a random 8-byte read costs what a 4-byte
// one does: 2.8 against 2.6 ns per wave and CU).  Per unit of slab area about
// 27 pixels are visited instead of 4 x 25 taps.  The transpose is the same
// gather with the windows' other bounds (|z - p_c| < 2 instead of the slab, no
// 5 x 5 windows, the mask on the pixels), where adj_lds_kernel spends half its
// time in 10 global atomics per pixel; its sums come in a fixed order.
//
// Work layout.  A wave owns 8 x 8 columns, bc_depth voxels long; the waves of
// a workgroup share them and take every fourth (eighth) direction each, into
// LDS accumulators of their own (lane-private columns: plain adds, no bank
// conflicts), combined in FP64 at the end.  The axis of the columns is that of
// the launch: three launches, one after the other, each taking the directions
// of its axis.  A wave handles one direction at a time, so the list of pixel
// offsets (from the pixel nearest to where the column meets the plane) is wave
// uniform and its position arithmetic reads the frame from scalar registers.
// The list holds every offset that can reach weight != 0 for some position of
// the crossing point inside its pixel: |u_a i + v_a j| <= 2 + (|u_a| + |v_a|) / 2
// for both cross axes a.
//
// Decisions are the reference's, each in its own FP32 arithmetic: the slab
// test, the rounded centre of every voxel's 5 x 5 window (a bit mask over the
// offsets per voxel) and the table indices.  The cross axes use kb_form's
// fused index (BP_FORM_A_MIN).  Along the column, slot k's index is slot 0's
// minus 125 k unless the FP32 rounding of the larger index value crosses a
// half-integer that the smaller one does not; then the larger one is exactly a
// half-integer (its spacing is at least the smaller one's and both are the
// same distance from theirs), so lanes that meet one take each slot's index by
// itself.
//
// Measured: 2,000 directions at N=128 6.9 (bp_fast_kernel) -> 6.3 ms, 1,000 at
// N=96 3.0 -> 2.0 ms; the transpose of 2,048 at N=96 6.5 -> 5.6 ms.  Bound by
// issue and LDS together: a pixel takes 37 vector instructions and five random
// table reads (13.6 ns per wave and CU of the 14.6 measured), and another 40%
// of the time goes to per-row and per-column work (windows, row bounds) at
// four waves per SIMD.  Blocks of 32 voxels (three waves per SIMD) ran 6.8 ms,
// four pixels at a time 7.0, one row buffer of three pixels with a compact
// loop 7.4.
// ---------------------------------------------------------------------------
constexpr int BCN = 8;                        // columns per block edge
// Voxels of a block along its columns: four (transpose: three) workgroups of
// four waves per CU.
constexpr int bc_depth(int mode) { return mode == COL_BACK ? 24 : 32; }

struct BPColArgs {
    BPArgs b;
    int blocks8;       // blocks along a cross axis
    int reachD2;       // largest squared distance from the centre of a voxel that is given values
};

__device__ __forceinline__ float read_lane_f(float x, int l)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l));
}

template <int MODE>
__device__ __forceinline__ float2 ct_pair(const float2 *__restrict__ st, int idx) { return st[idx - ct_lo(MODE)]; }

// One direction's visit of a wave's 64 columns, K slots per column.
// A: column axis (0, 1, 2 = x, y, z); the cross axes a, b are the others in
// order.  Vectors are in (a, b, c) order; onbits: slots that are active voxels;
// v0: first slot's coordinate along c.

template <int A, int K, int MODE>
struct ColVisit {
    static constexpr bool GATE = MODE == COL_BACK;
    // Back projection looks up p - v, the forward gather and so its transpose
    // v - p (a half-integer index rounds the other way).  The slots go along c
    // so that slot 0 has the largest index: up, or down.
    static constexpr int SG = GATE ? 1 : -1;
    static constexpr float SC = GATE ? 125.0f : -125.0f;

    static __device__ __forceinline__ float coord(float da, float db, float dc, float qa, float qb, float qc)
    {
        // ref_sum3 in x, y, z order
        if constexpr (A == 2) return ref_sum3(da, qa, db, qb, dc, qc);
        else if constexpr (A == 1) return ref_sum3(da, qa, dc, qc, db, qb);
        else return ref_sum3(dc, qc, da, qa, db, qb);
    }

    // half: half the extent along c of the voxels a column can be given values
    // in, from where it meets the plane.
    static __device__ __forceinline__ void run(
        const float2 *__restrict__ st, float *__restrict__ acc, const float *__restrict__ im,
        int M, int cv, int maskD2, int ln, float da, float db, int dzMax, int oc, int depth, int depthMax, float hw,
        float half, float ua, float ub, float uc, float va, float vb, float vc, float na, float nb, float nc)
    {
        const int ci = M / 2, M2 = M * M;
        const float cvf = (float)cv, cif = (float)ci;
        // where the column meets the plane, and its first voxel
        const float inv = __builtin_amdgcn_rcpf(nc);
        const float zc = -(na * da + nb * db) * inv;
        // relative to the volume's centre
        const int v0 = GATE ? (int)ceilf(zc - half - 5e-3f) : (int)floorf(zc + half + 5e-3f);
        const float fic = ua * da + ub * db + uc * zc, fjc = va * da + vb * db + vc * zc;
        int I0 = (int)rintf(fic), J0 = (int)rintf(fjc);

        unsigned onbits = 0;
        unsigned win[GATE ? K : 1];  // voxel k's 5 x 5 window: bits 8 + di low half, 8 + dj high half
        const int si0 = ci + I0 - 6, sj0 = ci + J0 - 22;
#pragma unroll
        for (int k = 0; k < K; k++) {
            const int dz = v0 + SG * k;
            bool on = (unsigned)(dz + cv - oc) < (unsigned)depth;
            if constexpr (GATE) {
                const float dc = (float)v0 + (float)k;
                const float fk = coord(da, db, dc, na, nb, nc);
                on = on && fabsf(fk) <= hw && abs(dz) <= dzMax;
                const float fi = coord(da, db, dc, ua, ub, uc) + cif;
                const float fj = coord(da, db, dc, va, vb, vc) + cif;
                // the window's centre is at most 3 pixels from (I0, J0) for
                // the slab's voxels
                const unsigned w = (0x1Fu << ((cvt_rpi(fi) - si0) & 31)) | (0x1Fu << ((cvt_rpi(fj) - sj0) & 31));
                win[k] = on ? w : 0u;
            }
            onbits |= on ? (1u << k) : 0u;
        }
        // Pixels that a column visits are within 9 of (I0, J0) in each index.
        const int ai = abs(I0), aj = abs(J0);
        if (!GATE && (dzMax < 0 || max(ai - 9, 0) * max(ai - 9, 0) + max(aj - 9, 0) * max(aj - 9, 0) > maskD2)) onbits = 0;
        const bool live = onbits != 0u;
        if (__ballot(live) == 0ull) return;
        // a column without a voxel to fill idles on the centre's
        const float ea = live ? da : 0.f, eb = live ? db : 0.f;
        const int e0c = live ? v0 : GATE ? (int)ceilf(-half - 5e-3f) : (int)floorf(half + 5e-3f);
        if (!live) I0 = J0 = 0;

        // Pixel offsets: lane r < 16 bounds row dj = r - 8 (rows with pixels are
        // consecutive).
        float rowLo = -8.f;
        int rowCnt;
        {
            const float dj = (float)((ln & 15) - 8);
            float hi = 7.f;
            auto bound = [&](float u, float v) {
                const float L = col_list_reach(u, v);
                if (fabsf(u) < 1e-6f) {
                    if (fabsf(v * dj) > L) hi = -9.f;
                } else {
                    const float r = __builtin_amdgcn_rcpf(u), p = (-L - v * dj) * r, q = (L - v * dj) * r;
                    rowLo = fmaxf(rowLo, ceilf(fminf(p, q)));
                    hi = fminf(hi, floorf(fmaxf(p, q)));
                }
            };
            bound(ua, va);
            bound(ub, vb);
            rowCnt = max((int)(hi - rowLo) + 1, 0);
        }
        const unsigned rows = (unsigned)__ballot(rowCnt > 0 && ln < 16);
        if (rows == 0u) return;
        int r = __builtin_ctz(rows);
        const int rEnd = 32 - __builtin_clz(rows);

        // index constants 250 -+ 125 v of the column and of its first slot
        const float cA = fmaf(-SC, ea + cvf, 250.0f), cB = fmaf(-SC, eb + cvf, 250.0f);
        const float cC = fmaf(-SC, (float)(e0c + cv), 250.0f);
        const int lin0 = (J0 + ci) * M + (I0 + ci);
        // every pixel of every lane is in the image (BACK) or the mask (ADJOINT)
        const bool allIn = GATE ? __all(lin0 >= 8 * M + 8 && lin0 + 8 * M + 14 <= M2)
                                : __all(!live || ((ai + 14) * (ai + 14) + (aj + 9) * (aj + 9) <= maskD2 &&
                                                  (ai + 14) * (ai + 14) <= maskD2));
        const float I0f = (float)I0;
        float djf = (float)(J0 + r - 8);

        float s[K];
#pragma unroll
        for (int k = 0; k < K; k++) s[k] = 0.f;

        // The values of six consecutive pixels from offset off (a row has five
        // on average).
        auto load = [&](int off, int row, int di, float (&x)[6]) {
            if (allIn) {
                const float *ip = (const float *)((const char *)(im + off) + (unsigned)lin0 * 4u);
                f4 q;
                __builtin_memcpy(&q, ip, 16);
                x[0] = q.x; x[1] = q.y; x[2] = q.z; x[3] = q.w;
                __builtin_memcpy(&x[4], ip + 4, 8);
            } else {
                // The reference's back projection bounds only the linear index
                // (gpuBackProject.cu:99): windows wrap across rows.  The
                // forward projection writes the pixels of the mask disc.
                const int dj = J0 + row - 8;
#pragma unroll
                for (int e = 0; e < 6; e++) {
                    const int lin = lin0 + off + e, i = I0 + di + e;
                    const bool ok = GATE ? lin >= 0 && lin < M2
                                         : i * i + dj * dj <= maskD2 && (unsigned)(i + ci) < (unsigned)M &&
                                               (unsigned)(dj + ci) < (unsigned)M;
                    const float raw = im[min(max(lin, 0), M2 - 1)];
                    x[e] = ok ? raw : 0.f;
                }
            }
        };
        // only the longest columns reach past the table's ends
        auto clampTo = [](bool on, int i) { return on ? min(max(i, ct_lo(MODE)), ct_hi(MODE) - 1) : i; };
        float Ba, Bb, Bc;
        unsigned eff[GATE ? K : 1];
        // NP pixels of the current row from offset di on (bit di + 8 of eff).
        auto pixels = [&](float Df, int di, const float *val, auto np) {
            constexpr int NP = decltype(np)::value;
            float wab[NP];
            float2 wc[NP][(K + 1) / 2];
            float sc[NP], pc[NP];
            bool tie = false;
#pragma unroll
            for (int q = 0; q < NP; q++) {
                const float Di = Df + (float)q;
                const float pa = fmaf(Di, ua, Ba) + cvf, pb = fmaf(Di, ub, Bb) + cvf;
                pc[q] = fmaf(Di, uc, Bc) + cvf;
                sc[q] = fmaf(pc[q], SC, cC);
                tie = tie || __builtin_amdgcn_fractf(sc[q]) == 0.5f;
                const int ic = cvt_rpi(sc[q]);
                wab[q] = ct_pair<MODE>(st, cvt_rpi(fmaf(pa, SC, cA))).x * ct_pair<MODE>(st, cvt_rpi(fmaf(pb, SC, cB))).x;
#pragma unroll
                for (int h = 0; h < (K + 1) / 2; h++) wc[q][h] = ct_pair<MODE>(st, clampTo(col_clamps(MODE, K), ic - 250 * h));
            }
            if (__any(tie)) {
#pragma unroll
                for (int q = 0; q < NP; q++)
#pragma unroll
                    for (int k = 0; k < K; k++) {
                        const int i = cvt_rpi(fmaf(pc[q], SC, cC - 125.0f * k));
                        float w = ct_pair<MODE>(st, clampTo(col_clamps_single(MODE, K), i)).x;
                        // keeps these loads apart from the paired ones (the
                        // compiler merges both into K single loads)
                        __asm__ volatile("" : "+v"(w));
                        if (k & 1) wc[q][k / 2].y = w; else wc[q][k / 2].x = w;
                    }
            }
#pragma unroll
            for (int q = 0; q < NP; q++) {
                const float wv = wab[q] * val[q];
#pragma unroll
                for (int k = 0; k < K; k++) {
                    float w = (k & 1) ? wc[q][k / 2].y : wc[q][k / 2].x;
                    if constexpr (GATE)
                        w = __int_as_float(__float_as_int(w) & __builtin_amdgcn_sbfe((int)eff[k], di + 8 + q, 1));
                    s[k] = fmaf(wv, w, s[k]);
                }
            }
        };
        // The next row's first six values are loaded while a row is gathered.
        float val[6];
        float lo = read_lane_f(rowLo, r);
        int cnt = __builtin_amdgcn_readlane(rowCnt, r), off = (r - 8) * M + (int)lo;
        load(off, r, (int)lo, val);
        while (true) {
            const float loN = read_lane_f(rowLo, r + 1);
            const int cntN = __builtin_amdgcn_readlane(rowCnt, r + 1), offN = (r - 7) * M + (int)loN;
            float nval[6];
            if (r + 1 < rEnd) load(offN, r + 1, (int)loN, nval);
            Ba = djf * va; Bb = djf * vb; Bc = djf * vc;
#pragma unroll
            for (int k = 0; k < (GATE ? K : 0); k++)
                eff[k] = win[k] & (unsigned)__builtin_amdgcn_sbfe((int)win[k], r + 16, 1);
            const float Df = I0f + lo;
            const int di = (int)lo;
            col_row(cnt, [&](auto first, auto np) {
                constexpr int F = decltype(first)::value;
                pixels(F ? Df + (float)F : Df, di + F, val + F, np);
            }, [&](int e, auto np) {
                float xv[6];
                load(off + e, r, di + e, xv);
                pixels(Df + (float)e, di + e, xv, np);
            });
            if (++r >= rEnd) break;
            lo = loN; cnt = cntN; off = offN;
            djf += 1.f;
#pragma unroll
            for (int e = 0; e < 6; e++) val[e] = nval[e];
        }
        // Slots that are no active voxel go to the accumulators' spare row.
        int row[K];
        float ov[K];
#pragma unroll
        for (int k = 0; k < K; k++) {
            row[k] = ((onbits >> k) & 1u ? v0 + SG * k + cv - oc : depthMax) * 64 + ln;
            ov[k] = acc[row[k]];
        }
#pragma unroll
        for (int k = 0; k < K; k++) acc[row[k]] = ov[k] + s[k];
        __asm__ volatile("" ::: "memory");
    }
};

template <int A, int MODE, int BCW>
__global__ __launch_bounds__(64 * BCW, MODE == COL_BACK ? 4 : 3) void col_kernel(BPColArgs p)
{
    constexpr bool GATE = MODE == COL_BACK;
    constexpr int D = bc_depth(MODE), LO = ct_lo(MODE), NT = ct_hi(MODE) - LO;
    __shared__ float2 st[NT];
    __shared__ float sacc[BCW][64 * (D + 1)];  // and a spare row

    // not set: the voxel (tile) kernel does it all
    if ((__builtin_amdgcn_readfirstlane(*p.b.check) & 1u) == 0u) return;
    const unsigned work = (unsigned)p.b.order[blockIdx.x];
    // block lattice (a, b, c), a fastest
    const int bc = (int)(work / (unsigned)(p.blocks8 * p.blocks8));
    const int rem = (int)(work - (unsigned)bc * (unsigned)(p.blocks8 * p.blocks8));
    const int bb = rem / p.blocks8, ba = rem - bb * p.blocks8;
    const int oa = ba * BCN, ob = bb * BCN, oc = bc * D;
    const int V = p.b.V, M = p.b.M, cv = V / 2;
    // Voxels farther from the centre than the mask radius (the transpose's
    // windows: 2 sqrt(3) more) take nothing.
    {
        auto gap = [&](int o, int e) { return max(max(o - cv, cv - (o + e - 1)), 0); };
        const int ga = gap(oa, BCN), gb = gap(ob, BCN), gc = gap(oc, D);
        if (ga * ga + gb * gb + gc * gc > p.reachD2) return;
    }
    const int t = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(t >> 6), ln = t & 63;
    for (int e = t; e < NT; e += 64 * BCW) {
        const int i = e + LO, j = i - 125;
        st[e] = make_float2(i >= 0 && i < KFAST ? p.b.ker[min(max(i, 0), KFAST - 1)] : 0.f,
                            j >= 0 && j < KFAST ? p.b.ker[min(max(j, 0), KFAST - 1)] : 0.f);
    }
    for (int e = t; e < BCW * 64 * (D + 1); e += 64 * BCW) (&sacc[0][0])[e] = 0.f;
    __syncthreads();

    const int depth = min(D, V - oc);
    // This lane's column, relative to the volume's centre, and how far the
    // mask sphere (the volume) reaches along it (-1: not at all).
    const int la = oa + (ln & 7) - cv, lb = ob + (ln >> 3) - cv;
    int dzMax = -1;
    if (oa + (ln & 7) < V && ob + (ln >> 3) < V) {
        const int rest = p.b.maskD2 - la * la - lb * lb;
        if (!GATE) {
            dzMax = V;
        } else if (rest >= 0) {
            dzMax = (int)sqrtf((float)rest);
            while (dzMax * dzMax > rest) dzMax--;
            while ((dzMax + 1) * (dzMax + 1) <= rest) dzMax++;
        }
    }
    const float da = (float)la, db = (float)lb;
    const float mA = (float)(oa - cv) + 0.5f * (BCN - 1), mB = (float)(ob - cv) + 0.5f * (BCN - 1);
    const float mC = (float)(oc - cv) + 0.5f * (D - 1);
    constexpr int ia = A == 0 ? 1 : 0, ib = A == 2 ? 1 : 2, ic = A;

    for (int base = 0; base < p.b.nAxes; base += BCW * 64) {
        const int mine = base + BCW * ln + wv;
        float a9[9];
        bool pass = false;
        if (mine < p.b.nAxes) {
            const float *ax = p.b.axes + (size_t)9 * mine;
#pragma unroll
            for (int k = 0; k < 9; k++) a9[k] = ax[k];
            const bool orth = GATE ? bp_orthonormal(a9, p.b.orthTol) : adj_plane(a9, p.b.orthTol);
            const float n0 = fabsf(a9[6 + ia]), n1 = fabsf(a9[6 + ib]), n2 = fabsf(a9[6 + ic]);
            // the launch whose axis is the normal's largest (the first of equals)
            const bool axis = (A == 0 ? n2 >= n0 : n2 > n0) && (A == 2 ? n2 > n1 : n2 >= n1);
            const float dist = mA * a9[6 + ia] + mB * a9[6 + ib] + mC * a9[6 + ic];
            const float reach = GATE ? p.b.hw : 2.f * (n0 + n1 + n2);  // a slab, or cubes of half edge 2
            pass = axis && orth && fabsf(dist) <= reach + 0.5f * (BCN - 1) * (n0 + n1) + 0.5f * (D - 1) * n2 + 1e-2f;
        } else {
#pragma unroll
            for (int k = 0; k < 9; k++) a9[k] = 0.f;
        }
        for (unsigned long long todo = __ballot(pass); todo != 0ull; todo &= todo - 1ull) {
            const int l = __builtin_ctzll(todo);
            const float ua = read_lane_f(a9[ia], l), ub = read_lane_f(a9[ib], l), uc = read_lane_f(a9[ic], l);
            const float va = read_lane_f(a9[3 + ia], l), vb = read_lane_f(a9[3 + ib], l), vc = read_lane_f(a9[3 + ic], l);
            const float na = read_lane_f(a9[6 + ia], l), nb = read_lane_f(a9[6 + ib], l), nc = read_lane_f(a9[6 + ic], l);
            const float *im = p.b.img + (size_t)(base + BCW * l + wv) * M * M;
            // A column's voxels: |fk| <= 2, or (transpose) |z - p_c| < 2 of a
            // pixel with |p_a - x_a|, |p_b - x_b| < 2: at most
            // floor(2 half) + 1 consecutive ones.
            const float half = (GATE ? p.b.hw : 2.f * (fabsf(na) + fabsf(nb) + fabsf(nc))) *
                               __builtin_amdgcn_rcpf(fabsf(nc));
            const float len = 2.f * half + 1.5e-2f;
#define MGG_VISIT(KS) ColVisit<A, KS, MODE>::run(st, sacc[wv], im, M, cv, p.b.maskD2, ln, da, \
                                                       db, dzMax, oc, depth, D, p.b.hw, half, ua, ub, uc, va, vb, \
                                                       vc, na, nb, nc)
            const int slots = __builtin_amdgcn_readfirstlane(col_slots(MODE, len));
            if constexpr (GATE) {
                if (slots == 5) MGG_VISIT(5);
                else if (slots == 6) MGG_VISIT(6);
                else MGG_VISIT(7);
            } else {
                if (slots == 6) MGG_VISIT(6);
                else if (slots == 8) MGG_VISIT(8);
                else if (slots == 10) MGG_VISIT(10);
                else MGG_VISIT(14);
            }
#undef MGG_VISIT
        }
    }
    __syncthreads();
    // Add to the volume, x fastest: the columns' layout is [c][b][a].
    for (int e = t; e < 64 * D; e += 64 * BCW) {
        int qa, qb, qc;
        if (A == 0) { qc = e % D; qa = (e / D) & 7; qb = e / (8 * D); }
        else { qa = e & 7; qb = (e >> 3) & 7; qc = e >> 6; }
        const int xa = oa + qa, xb = ob + qb, xc = oc + qc;
        if (xa >= V || xb >= V || xc >= V) continue;
        const int d2 = (xa - cv) * (xa - cv) + (xb - cv) * (xb - cv) + (xc - cv) * (xc - cv);
        if (d2 > p.reachD2) continue;
        const int x = A == 0 ? xc : xa, y = A == 0 ? xa : A == 1 ? xc : xb, z = A == 2 ? xc : xb;
        const size_t vidx = ((size_t)z * V + y) * V + x;
        const int slot = qc * 64 + qb * 8 + qa;
        double sum = (double)p.b.vol[vidx];
#pragma unroll
        for (int w = 0; w < BCW; w++) sum += (double)sacc[w][slot];
        p.b.vol[vidx] = (float)sum;
    }
}

// ---------------------------------------------------------------------------
// Image chains.  With even M, fftshift o DFT o fftshift equals the plain DFT
// with a (-1)^(x+y) checkerboard on input and output (the 2-D global sign
// (-1)^M is +1), so the shifts of gpuGridder.cpp:463-488 and :562-587 fold
// into these loads and stores.  The CAS-derived spectrum is exactly Hermitian,
// so the inverse uses C2R and the forward R2C (half the FFT work).
// ---------------------------------------------------------------------------
__device__ __forceinline__ float chk(int s) { return (s & 1) ? -1.f : 1.f; }

// The 2-D chain kernels run one workgroup per (row, image): blockIdx.x is the
// row, blockIdx.y strides over the images, the threads over the row, so every
// index is 32-bit arithmetic on the row and column (no per-element division)
// and each row is read and written contiguously.

// CASToComplexFilter.cu:53-75 (2-D stack mode) + fftshift, half spectrum.
__global__ void k_cas_to_herm2d(const float *__restrict__ cas, float2 *__restrict__ herm, int M, int n)
{
    const int H = M / 2 + 1;
    const int cy = blockIdx.x;
    for (int a = blockIdx.y; a < n; a += gridDim.y) {
        const float *c = cas + (size_t)a * M * M;
        float2 *h = herm + ((size_t)a * M + cy) * H;
        for (int cx = threadIdx.x; cx < H; cx += blockDim.x) {
            float2 z = make_float2(0.f, 0.f);
            if (cx != 0 && cy != 0) {
                const float c1 = c[cy * M + cx];
                const float c2 = c[(M - cy) * M + (M - cx)];
                const float sg = chk(cx + cy);
                z.x = sg * (0.5f * (c1 + c2));
                z.y = sg * (0.5f * (c1 - c2));
            }
            h[cx] = z;
        }
    }
}

// fftshift + ComplexToReal + CropVolume + DivideScalar (gpuGridder.cpp:485-517).
__global__ void k_real2d_to_imgs(const float *__restrict__ real, float *__restrict__ imgs, int M,
                                 int N, float scale, int n)
{
    const int off = (M - N) / 2;
    const int py = blockIdx.x, my = py + off;
    for (int a = blockIdx.y; a < n; a += gridDim.y) {
        const float *r = real + ((size_t)a * M + my) * M + off;
        float *o = imgs + ((size_t)a * N + py) * N;
        for (int px = threadIdx.x; px < N; px += blockDim.x)
            o[px] = chk(px + off + my) * r[px] * scale;
    }
}

// PadVolume + RealToComplex + fftshift (gpuGridder.cpp:543-566).
__global__ void k_imgs_to_real2d(const float *__restrict__ imgs, float *__restrict__ real, int M,
                                 int N, int n)
{
    const int off = (M - N) / 2;
    const int my = blockIdx.x, py = my - off;
    const bool rowIn = py >= 0 && py < N;
    for (int a = blockIdx.y; a < n; a += gridDim.y) {
        const float *im = imgs + ((size_t)a * N + (rowIn ? py : 0)) * N;
        float *o = real + ((size_t)a * M + my) * M;
        for (int mx = threadIdx.x; mx < M; mx += blockDim.x) {
            const int px = mx - off;
            float v = 0.f;
            if (rowIn && px >= 0 && px < N) v = chk(mx + my) * im[px];
            o[mx] = v;
        }
    }
}

// fftshift + ComplexToCAS (gpuGridder.cpp:584-595) from the R2C half spectrum.
__global__ void k_herm2d_to_cas(const float2 *__restrict__ herm, float *__restrict__ cas, int M, int n,
                                float scale, int zeroNyq)
{
    const int H = M / 2 + 1;
    const int cy = blockIdx.x, my = (M - cy) % M;
    for (int a = blockIdx.y; a < n; a += gridDim.y) {
        const float2 *h = herm + (size_t)a * M * H;
        const float2 *hr = h + (size_t)cy * H, *hm = h + (size_t)my * H;
        float *o = cas + ((size_t)a * M + cy) * M;
        for (int cx = threadIdx.x; cx < M; cx += blockDim.x) {
            float re, im;
            if (cx <= M / 2) {
                const float2 f = hr[cx];
                re = f.x; im = f.y;
            } else {
                const float2 f = hm[M - cx];
                re = f.x; im = -f.y;
            }
            const float sg = chk(cx + cy);
            // zeroNyq: the index-0 row / column FromCAS discards (transpose of
            // the inverse image chain); scale is exact (1) on the forward chain.
            o[cx] = (zeroNyq && (cx == 0 || cy == 0)) ? 0.f : (sg * re + sg * im) * scale;
        }
    }
}

// ---------------------------------------------------------------------------
// Fused image chains for M = 128, 192, 256, 384 and 512.  The general chains above make
// five or six HBM passes per image (CAS -> Hermitian half spectrum, two rocFFT
// passes, crop; or the reverse).  These make two each, with the M-point FFT
// done in LDS as four-step 16 x R (M = 16 R; 16 threads per transform, the
// R-point and 16-point DFTs in registers, one twiddled exchange through LDS;
// the 32-point DFT is two 16-point DFTs and a radix-2 step, the 8-point DFT
// two 4-point DFTs and a radix-2 step, the 12- and 24-point DFTs 4- and
// 8-point DFTs and a radix-3 step), and are ordered
// so that CAS images are read and written as whole rows:
//   CAS images -> images: (1) k_inv_rows: per spectrum row ky <= M/2 the full
//   complex row is built from CAS rows ky and M - ky as they are read,
//   inverse-transformed along x, and the N cropped columns are kept
//   ((M/2 + 1) x N complex per image; rows ky > M/2 follow by Hermitian
//   symmetry); (2) k_inv_cols: 32 columns per workgroup, two Hermitian
//   columns per complex transform along y (its real and imaginary outputs are
//   the two real columns), checkerboard and 1/M^2, written through LDS.
//   images -> CAS images: (1) k_fwd_cols: two zero-padded image columns per
//   complex transform along y, split into two half spectra; (2) k_fwd_rows:
//   per spectrum row ky <= M/2 the transform along x gives the full row, and
//   CAS rows ky and M - ky are written whole.
// Same arithmetic as the general chains up to FP32 rounding in the FFT
// (twiddles from sincospif, accurate to ~1 ulp).
// ---------------------------------------------------------------------------
struct F16Tw { float c, s; };
__device__ __constant__ const F16Tw kTw16[16] = {
    {1.0f, 0.0f},
    {0.92387953251128674f, 0.38268343236508977f},
    {0.70710678118654752f, 0.70710678118654752f},
    {0.38268343236508977f, 0.92387953251128674f},
    {0.0f, 1.0f},
    {-0.38268343236508977f, 0.92387953251128674f},
    {-0.70710678118654752f, 0.70710678118654752f},
    {-0.92387953251128674f, 0.38268343236508977f},
    {-1.0f, 0.0f},
    {-0.92387953251128674f, -0.38268343236508977f},
    {-0.70710678118654752f, -0.70710678118654752f},
    {-0.38268343236508977f, -0.92387953251128674f},
    {0.0f, -1.0f},
    {0.38268343236508977f, -0.92387953251128674f},
    {0.70710678118654752f, -0.70710678118654752f},
    {0.92387953251128674f, -0.38268343236508977f}};

__device__ __forceinline__ float2 cmulw(float2 a, float c, float s)
{
    return make_float2(fmaf(a.x, c, -a.y * s), fmaf(a.x, s, a.y * c));
}

// 4-point DFT in place, X[k] = sum_n x[n] e^{S 2 pi i n k / 4}.
template <int S>
__device__ __forceinline__ void fft4(float2 &a, float2 &b, float2 &c, float2 &d)
{
    const float2 t0 = make_float2(a.x + c.x, a.y + c.y), t1 = make_float2(a.x - c.x, a.y - c.y);
    const float2 t2 = make_float2(b.x + d.x, b.y + d.y), t3 = make_float2(b.x - d.x, b.y - d.y);
    const float2 r = S > 0 ? make_float2(-t3.y, t3.x) : make_float2(t3.y, -t3.x);
    a = make_float2(t0.x + t2.x, t0.y + t2.y);
    c = make_float2(t0.x - t2.x, t0.y - t2.y);
    b = make_float2(t1.x + r.x, t1.y + r.y);
    d = make_float2(t1.x - r.x, t1.y - r.y);
}

// 16-point DFT in registers (radix 4 x 4).  Input v[n] in natural order;
// output X[k2 + 4 k1] is left in v[4 k2 + k1].
template <int S>
__device__ __forceinline__ void fft16(float2 (&v)[16])
{
#pragma unroll
    for (int n1 = 0; n1 < 4; n1++) fft4<S>(v[n1], v[n1 + 4], v[n1 + 8], v[n1 + 12]);
#pragma unroll
    for (int n1 = 1; n1 < 4; n1++)
#pragma unroll
        for (int k2 = 1; k2 < 4; k2++) {
            const F16Tw w = kTw16[n1 * k2];
            v[n1 + 4 * k2] = cmulw(v[n1 + 4 * k2], w.c, S > 0 ? w.s : -w.s);
        }
#pragma unroll
    for (int k2 = 0; k2 < 4; k2++) fft4<S>(v[4 * k2], v[4 * k2 + 1], v[4 * k2 + 2], v[4 * k2 + 3]);
}

__device__ __forceinline__ constexpr int fft16_slot(int k) { return 4 * (k & 3) + (k >> 2); }

// cos, sin of 2 pi j / 32, j = 0..15
__device__ __constant__ const F16Tw kTw32[16] = {
    {1.0f, 0.0f},
    {0.98078528040323043f, 0.19509032201612825f},
    {0.92387953251128674f, 0.38268343236508977f},
    {0.83146961230254524f, 0.55557023301960218f},
    {0.70710678118654752f, 0.70710678118654752f},
    {0.55557023301960218f, 0.83146961230254524f},
    {0.38268343236508977f, 0.92387953251128674f},
    {0.19509032201612825f, 0.98078528040323043f},
    {0.0f, 1.0f},
    {-0.19509032201612825f, 0.98078528040323043f},
    {-0.38268343236508977f, 0.92387953251128674f},
    {-0.55557023301960218f, 0.83146961230254524f},
    {-0.70710678118654752f, 0.70710678118654752f},
    {-0.83146961230254524f, 0.55557023301960218f},
    {-0.92387953251128674f, 0.38268343236508977f},
    {-0.98078528040323043f, 0.19509032201612825f}};

// 32-point DFT in registers: two 16-point DFTs (even and odd inputs) and a
// radix-2 combination.  X[k] is left in v[fft16_slot(k)], X[k + 16] in
// v[16 + fft16_slot(k)].
template <int S>
__device__ __forceinline__ void fft32(float2 (&v)[32])
{
    float2 e[16], o[16];
#pragma unroll
    for (int i = 0; i < 16; i++) {
        e[i] = v[2 * i];
        o[i] = v[2 * i + 1];
    }
    fft16<S>(e);
    fft16<S>(o);
#pragma unroll
    for (int k = 0; k < 16; k++) {
        const F16Tw w = kTw32[k];
        const float2 E = e[fft16_slot(k)], O = cmulw(o[fft16_slot(k)], w.c, S > 0 ? w.s : -w.s);
        v[fft16_slot(k)] = make_float2(E.x + O.x, E.y + O.y);
        v[16 + fft16_slot(k)] = make_float2(E.x - O.x, E.y - O.y);
    }
}

// 8-point DFT in registers: two 4-point DFTs (even and odd inputs) and a
// radix-2 combination; input and output in natural order.
template <int S>
__device__ __forceinline__ void fft8(float2 (&v)[8])
{
    float2 e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6];
    float2 o0 = v[1], o1 = v[3], o2 = v[5], o3 = v[7];
    fft4<S>(e0, e1, e2, e3);
    fft4<S>(o0, o1, o2, o3);
    constexpr float h = 0.70710678118654752f;  // cos(pi / 4)
    o1 = cmulw(o1, h, S > 0 ? h : -h);
    o2 = S > 0 ? make_float2(-o2.y, o2.x) : make_float2(o2.y, -o2.x);
    o3 = cmulw(o3, -h, S > 0 ? h : -h);
    v[0] = make_float2(e0.x + o0.x, e0.y + o0.y);
    v[4] = make_float2(e0.x - o0.x, e0.y - o0.y);
    v[1] = make_float2(e1.x + o1.x, e1.y + o1.y);
    v[5] = make_float2(e1.x - o1.x, e1.y - o1.y);
    v[2] = make_float2(e2.x + o2.x, e2.y + o2.y);
    v[6] = make_float2(e2.x - o2.x, e2.y - o2.y);
    v[3] = make_float2(e3.x + o3.x, e3.y + o3.y);
    v[7] = make_float2(e3.x - o3.x, e3.y - o3.y);
}

// cos, sin of 2 pi j / 24, j = 0..14
__device__ __constant__ const F16Tw kTw24[15] = {
    {1.00000000000000000f, 0.00000000000000000f},
    {0.96592582628906831f, 0.25881904510252074f},
    {0.86602540378443871f, 0.49999999999999994f},
    {0.70710678118654757f, 0.70710678118654746f},
    {0.50000000000000011f, 0.86602540378443860f},
    {0.25881904510252074f, 0.96592582628906831f},
    {0.00000000000000006f, 1.00000000000000000f},
    {-0.25881904510252063f, 0.96592582628906831f},
    {-0.49999999999999978f, 0.86602540378443871f},
    {-0.70710678118654746f, 0.70710678118654757f},
    {-0.86602540378443871f, 0.49999999999999994f},
    {-0.96592582628906820f, 0.25881904510252102f},
    {-1.00000000000000000f, 0.00000000000000012f},
    {-0.96592582628906831f, -0.25881904510252079f},
    {-0.86602540378443882f, -0.49999999999999972f}};

// 3-point DFT in place (natural order).
template <int S>
__device__ __forceinline__ void fft3(float2 &a, float2 &b, float2 &c)
{
    constexpr float s3 = 0.86602540378443865f;  // sin(2 pi / 3)
    const float2 t1 = make_float2(b.x + c.x, b.y + c.y);
    const float2 t2 = make_float2(a.x - 0.5f * t1.x, a.y - 0.5f * t1.y);
    const float2 d = make_float2(b.x - c.x, b.y - c.y);
    const float2 r = S > 0 ? make_float2(-s3 * d.y, s3 * d.x) : make_float2(s3 * d.y, -s3 * d.x);
    a = make_float2(a.x + t1.x, a.y + t1.y);
    b = make_float2(t2.x + r.x, t2.y + r.y);
    c = make_float2(t2.x - r.x, t2.y - r.y);
}

// 12- and 24-point DFTs in registers, natural order in and out: n = 3 p + q,
// k = k1 + (R / 3) k2; a (R / 3)-point DFT over p for each q, twiddles
// w_R^(q k1), then a 3-point DFT over q for each k1.
template <int S>
__device__ __forceinline__ void fft12(float2 (&v)[12])
{
    float2 b[3][4];
#pragma unroll
    for (int q = 0; q < 3; q++) {
        float2 a0 = v[q], a1 = v[3 + q], a2 = v[6 + q], a3 = v[9 + q];
        fft4<S>(a0, a1, a2, a3);
        b[q][0] = a0; b[q][1] = a1; b[q][2] = a2; b[q][3] = a3;
#pragma unroll
        for (int k1 = 1; k1 < 4; k1++) {
            if (q == 0) continue;
            const F16Tw w = kTw24[2 * q * k1];
            b[q][k1] = cmulw(b[q][k1], w.c, S > 0 ? w.s : -w.s);
        }
    }
#pragma unroll
    for (int k1 = 0; k1 < 4; k1++) {
        float2 x0 = b[0][k1], x1 = b[1][k1], x2 = b[2][k1];
        fft3<S>(x0, x1, x2);
        v[k1] = x0; v[k1 + 4] = x1; v[k1 + 8] = x2;
    }
}

template <int S>
__device__ __forceinline__ void fft24(float2 (&v)[24])
{
    float2 b[3][8];
#pragma unroll
    for (int q = 0; q < 3; q++) {
#pragma unroll
        for (int p8 = 0; p8 < 8; p8++) b[q][p8] = v[3 * p8 + q];
        fft8<S>(b[q]);
#pragma unroll
        for (int k1 = 1; k1 < 8; k1++) {
            if (q == 0) continue;
            const F16Tw w = kTw24[q * k1];
            b[q][k1] = cmulw(b[q][k1], w.c, S > 0 ? w.s : -w.s);
        }
    }
#pragma unroll
    for (int k1 = 0; k1 < 8; k1++) {
        float2 x0 = b[0][k1], x1 = b[1][k1], x2 = b[2][k1];
        fft3<S>(x0, x1, x2);
        v[k1] = x0; v[k1 + 8] = x1; v[k1 + 16] = x2;
    }
}

template <int R, int S>
__device__ __forceinline__ void fft_regs(float2 (&v)[R])
{
    if constexpr (R == 8) fft8<S>(v);
    else if constexpr (R == 12) fft12<S>(v);
    else if constexpr (R == 16) fft16<S>(v);
    else if constexpr (R == 24) fft24<S>(v);
    else fft32<S>(v);
}

// Position of X[k] in v[] after fft_regs<R>.
template <int R>
__device__ __forceinline__ constexpr int fftR_slot(int k)
{
    return (R == 8 || R == 12 || R == 24) ? k
         : (R == 16 ? fft16_slot(k) : (k < 16 ? fft16_slot(k) : 16 + fft16_slot(k - 16)));
}

// After fft_m<R>, thread t holds X[out_idx<R>(t, m)] in v[out_slot<R>(m)],
// m < R (see there).
template <int R>
__device__ __forceinline__ constexpr int out_slot(int m)
{
    return (R == 8 || R == 12 || R == 24) ? m : (R == 16 ? fft16_slot(m) : 16 * (m & 1) + fft16_slot(m >> 1));
}

template <int R>
__device__ __forceinline__ int out_idx(int t, int m)
{
    if constexpr (R == 12 || R == 24) {
        constexpr int D = R == 12 ? 4 : 2, L = 16 / D;
        const int P = t + 16 * (m / L), mm = m % L;
        return P % R + R * (D * mm + P / R);
    } else {
        return t + 16 * m;
    }
}

// Index of the mirrored row or column, (M - k) mod M, for 0 <= k < M.
template <int M>
__device__ __forceinline__ int mirror_idx(int k)
{
    if constexpr ((M & (M - 1)) == 0) return (M - k) & (M - 1);
    else return k == 0 ? 0 : M - k;
}

constexpr int FFP = 17;  // exchange pitch (float2)
template <int R> struct FftGeom {
    static constexpr int M = 16 * R, H = M / 2 + 1;
    // LDS float2 per transform (>= M); the odd extra float2 puts the
    // transforms of a workgroup on different banks, where 16 * 17 * 2 floats
    // (0 mod 32) put them all on one (the column fills write one element of
    // each of 16 transforms per row; 3-5% faster chains at M = 256).
    static constexpr int FFB = R * FFP + 1;
};

// M-point DFT (M = 16 R) by the 16 threads t = 0..15 of one transform,
// four-step 16 x R: R-point DFTs in registers, twiddles, exchange through
// LDS, 16-point DFTs (outputs X[k2 + R k1], k2 < R, k1 < 16).  On entry v[n2]
// holds x[t + 16 n2] (n2 < R); on exit v[out_slot<R>(m)] holds
// X[out_idx<R>(t, m)] (m < R).  With R = 16, 32 thread t does the 16-point
// DFTs of k2 = t + 16 j (out_idx = t + 16 m).  Otherwise each 16-point DFT is
// shared by D threads through one radix-D decimation in frequency: the share
// h < D takes the outputs k1 = D mm + h, an L = 16 / D point DFT over n of
// w16^(n h) sum_e z[n + L e] w_D^(e h).  R = 8: D = 2, thread t takes
// k2 = t % 8, h = t / 8 (out_idx = t + 16 m again); R = 12 (D = 4) and
// R = 24 (D = 2): thread t takes the three (k2, h) = (P % R, P / R),
// P = t + 16 j, j < 3.
// ex is the transform's FFB-float2 LDS exchange area, tw the M twiddles
// e^{2 pi i q / M}.  Contains workgroup barriers: every thread of the block
// must call it.
template <int R, int S>
__device__ __forceinline__ void fft_m(float2 (&v)[R], int t, float2 *ex, const float2 *tw)
{
    fft_regs<R, S>(v);
#pragma unroll
    for (int k2 = 0; k2 < R; k2++) {
        const float2 w = tw[t * k2];
        ex[k2 * FFP + t] = cmulw(v[fftR_slot<R>(k2)], w.x, S > 0 ? w.y : -w.y);
    }
    __syncthreads();
    if constexpr (R == 8) {
        const int k2 = t & 7, hf = t >> 3;
        const float sg = hf ? -1.f : 1.f;
#pragma unroll
        for (int n = 0; n < 8; n++) {
            const float2 z0 = ex[k2 * FFP + n], z1 = ex[k2 * FFP + n + 8];
            const float2 d = make_float2(fmaf(sg, z1.x, z0.x), fmaf(sg, z1.y, z0.y));
            const float2 w = tw[((16 * R) / 16) * n * hf];  // w16^(n h)
            v[n] = cmulw(d, w.x, S > 0 ? w.y : -w.y);
        }
        fft8<S>(v);
    } else if constexpr (R == 12 || R == 24) {
        constexpr int D = R == 12 ? 4 : 2, L = 16 / D;
#pragma unroll
        for (int j = 0; j < 3; j++) {
            const int P = t + 16 * j, k2 = P % R, h = P / R;
            float2 b[L];
#pragma unroll
            for (int n = 0; n < L; n++) {
                float2 sm;
                if constexpr (D == 2) {
                    const float2 z0 = ex[k2 * FFP + n], z1 = ex[k2 * FFP + n + 8];
                    const float sg = h ? -1.f : 1.f;
                    sm = make_float2(fmaf(sg, z1.x, z0.x), fmaf(sg, z1.y, z0.y));
                } else {
                    sm = ex[k2 * FFP + n];
#pragma unroll
                    for (int e = 1; e < 4; e++) {
                        // z * (S i)^(e h): quarter turns, counter-clockwise for S > 0
                        const float2 z = ex[k2 * FFP + n + 4 * e];
                        const int ph = (S > 0 ? e * h : 4 * e - e * h) & 3;
                        const float2 r = ph == 0 ? z : ph == 1 ? make_float2(-z.y, z.x)
                                       : ph == 2 ? make_float2(-z.x, -z.y) : make_float2(z.y, -z.x);
                        sm = make_float2(sm.x + r.x, sm.y + r.y);
                    }
                }
                const float2 w = tw[R * n * h];  // w16^(n h)
                b[n] = cmulw(sm, w.x, S > 0 ? w.y : -w.y);
            }
            if constexpr (L == 4) fft4<S>(b[0], b[1], b[2], b[3]);
            else fft8<S>(b);
#pragma unroll
            for (int mm = 0; mm < L; mm++) v[j * L + mm] = b[mm];
        }
    } else {
#pragma unroll
        for (int j = 0; j < R / 16; j++) {
            float2 u[16];
#pragma unroll
            for (int n1 = 0; n1 < 16; n1++) u[n1] = ex[(t + 16 * j) * FFP + n1];
            fft16<S>(u);
#pragma unroll
            for (int q = 0; q < 16; q++) v[16 * j + q] = u[q];
        }
    }
    __syncthreads();  // the exchange area may be reused
}

template <int R>
__device__ __forceinline__ void load_tw(float2 *tw)
{
    constexpr int M = 16 * R;
    for (int q = threadIdx.x; q < M; q += blockDim.x) {
        float sn, cs;
        sincospif((float)q / (float)(M / 2), &sn, &cs);
        tw[q] = make_float2(cs, sn);
    }
}

// CAS images -> R[a][ky][mx'] (ky in [0, M/2 + 1), mx' in [0, N)): per spectrum
// row ky the full complex row is built from CAS rows ky and M - ky as they are
// read (whole rows), transformed along x, and the N kept columns are stored.
// Rows ky > M/2 are not needed: R[M - ky] = conj R[ky].  Grid (row groups of
// 16, images).
template <int R>
__global__ __launch_bounds__(256) void k_inv_rows(const float *__restrict__ cas, float2 *__restrict__ tmp,
                                                  int n, int N)
{
    using G = FftGeom<R>;
    constexpr int M = G::M, H = G::H;
    __shared__ float2 sx[16 * G::FFB];
    __shared__ float2 tw[M];
    load_tw<R>(tw);
    const int tid = threadIdx.x, f = tid >> 4, t = tid & 15;
    const int off = (M - N) / 2;
    const int ky = 16 * blockIdx.x + f;
    const bool rowOk = ky <= M / 2;
    float2 *ex = sx + f * G::FFB;
    for (int a = blockIdx.y; a < n; a += gridDim.y) {
        const float *rowA = cas + (size_t)a * M * M + (size_t)(rowOk ? ky : 0) * M;
        const float *rowB = cas + (size_t)a * M * M + (size_t)mirror_idx<M>(ky) * M;
        // Unconditional loads (every address is inside the image), so that all
        // 2R are in flight before the first use; the CAS index 0 row and column
        // select zero afterwards (rows beyond M/2 are not stored).
        float c1[R], c2[R];
#pragma unroll
        for (int n2 = 0; n2 < R; n2++) {
            const int kx = t + 16 * n2;
            c1[n2] = rowA[kx];
            c2[n2] = rowB[mirror_idx<M>(kx)];
        }
        float2 v[R];
#pragma unroll
        for (int n2 = 0; n2 < R; n2++) {
            const int kx = t + 16 * n2;
            const float sg = chk(kx + ky);
            v[n2] = make_float2(sg * (0.5f * (c1[n2] + c2[n2])), sg * (0.5f * (c1[n2] - c2[n2])));
        }
        if (t == 0) v[0] = make_float2(0.f, 0.f);  // kx = 0, NaN included
        if (ky == 0) {
#pragma unroll
            for (int n2 = 0; n2 < R; n2++) v[n2] = make_float2(0.f, 0.f);
        }
        __syncthreads();
        fft_m<R, 1>(v, t, ex, tw);
        if (rowOk) {
            float2 *o = tmp + ((size_t)a * H + ky) * N;
#pragma unroll
            for (int m = 0; m < R; m++) {
                const int px = out_idx<R>(t, m) - off;
                if (px >= 0 && px < N) o[px] = v[out_slot<R>(m)];
            }
        }
    }
}

// R -> images: 32 columns per workgroup, two Hermitian columns packed into one
// complex transform along y (its real and imaginary outputs are the two real
// columns); output through LDS as whole row segments.  Grid (ceil(N / 32),
// images).
template <int R>
__global__ __launch_bounds__(256) void k_inv_cols(const float2 *__restrict__ tmp, float *__restrict__ imgs,
                                                  int n, int N, float scale)
{
    using G = FftGeom<R>;
    constexpr int M = G::M, H = G::H;
    __shared__ float2 sx[16 * G::FFB];
    __shared__ float2 tw[M];
    load_tw<R>(tw);
    const int tid = threadIdx.x, f = tid >> 4, t = tid & 15;
    const int off = (M - N) / 2;
    const int c0 = 32 * blockIdx.x;
    float2 *ex = sx + f * G::FFB;
    float *so = reinterpret_cast<float *>(sx);  // output staging, pitch 33 floats (N * 33 <= 32 * FFB)
    for (int a = blockIdx.y; a < n; a += gridDim.y) {
        __syncthreads();
        // Z_f[ky] = R[ky][c0 + 2f] + i R[ky][c0 + 2f + 1], and by symmetry
        // Z_f[M - ky] = conj R[ky][2f] + i conj R[ky][2f + 1].  Eight loads per
        // thread in flight before the first exchange and LDS store (lanes 2j
        // and 2j + 1 hold neighbouring columns of one row: both in range or
        // both not, since H * 32 is even).
        constexpr int LB = 8;
        for (int base = tid; base < H * 32; base += 256 * LB) {
            float2 vals[LB];
#pragma unroll
            for (int q = 0; q < LB; q++) {
                // unconditional load from a clamped (in-range) address
                const int idx = base + 256 * q, ky = idx >> 5, px = c0 + (idx & 31);
                const float2 raw = tmp[((size_t)a * H + min(ky, H - 1)) * N + min(px, N - 1)];
                vals[q] = (idx < H * 32 && px < N) ? raw : make_float2(0.f, 0.f);
            }
#pragma unroll
            for (int q = 0; q < LB; q++) {
                const int idx = base + 256 * q, ky = idx >> 5, col = idx & 31;
                const float2 val = vals[q];
                const float ox = __shfl_xor(val.x, 1), oy = __shfl_xor(val.y, 1);
                if (idx < H * 32 && !(col & 1)) {
                    float2 *zf = sx + (col >> 1) * G::FFB;
                    zf[ky] = make_float2(val.x - oy, val.y + ox);
                    if (ky != 0 && ky != M / 2) zf[M - ky] = make_float2(val.x + oy, ox - val.y);
                }
            }
        }
        __syncthreads();
        float2 v[R];
#pragma unroll
        for (int n2 = 0; n2 < R; n2++) v[n2] = ex[t + 16 * n2];
        __syncthreads();
        fft_m<R, 1>(v, t, ex, tw);
#pragma unroll
        for (int m = 0; m < R; m++) {
                const int my = out_idx<R>(t, m), py = my - off;
                if (py >= 0 && py < N) {
                    const float2 z = v[out_slot<R>(m)];
                    const int mx = c0 + 2 * f + off;
                    so[py * 33 + 2 * f] = chk(mx + my) * z.x * scale;
                    so[py * 33 + 2 * f + 1] = chk(mx + 1 + my) * z.y * scale;
                }
            }
        __syncthreads();
        for (int idx = tid; idx < N * 32; idx += 256) {
            const int py = idx >> 5, col = idx & 31, px = c0 + col;
            if (px < N) imgs[((size_t)a * N + py) * N + px] = so[py * 33 + col];
        }
    }
}

// Images -> C[a][ky][px] (ky in [0, M/2 + 1)): 32 image columns per workgroup,
// two zero-padded real columns per complex transform along y, split into the
// two half spectra; input through LDS from whole row segments.  Grid
// (ceil(N / 32), images).
template <int R>
__global__ __launch_bounds__(256) void k_fwd_cols(const float *__restrict__ imgs, float2 *__restrict__ tmp,
                                                  int n, int N)
{
    using G = FftGeom<R>;
    constexpr int M = G::M, H = G::H;
    __shared__ float2 sx[16 * G::FFB];
    __shared__ float2 tw[M];
    load_tw<R>(tw);
    const int tid = threadIdx.x, f = tid >> 4, t = tid & 15;
    const int off = (M - N) / 2;
    const int c0 = 32 * blockIdx.x;
    float2 *ex = sx + f * G::FFB;
    float *sf = reinterpret_cast<float *>(sx);
    for (int a = blockIdx.y; a < n; a += gridDim.y) {
        __syncthreads();
        // Column c0 + col goes to transform col / 2, real (even) or imaginary
        // part.  The N image rows are loaded eight per thread at a time, all
        // eight in flight before the first LDS store; the M - N padding rows
        // are zeros.
        constexpr int LB = 8;
        for (int base = tid; base < N * 32; base += 256 * LB) {
            float xv[LB];
#pragma unroll
            for (int q = 0; q < LB; q++) {
                // unconditional load from a clamped (in-image) address, so that
                // no branch separates the eight loads
                const int idx = base + 256 * q, py = idx >> 5, col = idx & 31, px = c0 + col;
                const float raw = imgs[((size_t)a * N + min(py, N - 1)) * N + min(px, N - 1)];
                xv[q] = (idx < N * 32 && px < N) ? chk(px + off + py + off) * raw : 0.f;
            }
#pragma unroll
            for (int q = 0; q < LB; q++) {
                const int idx = base + 256 * q, col = idx & 31;
                if (idx < N * 32) sf[((col >> 1) * G::FFB + (idx >> 5) + off) * 2 + (col & 1)] = xv[q];
            }
        }
        for (int idx = tid; idx < (M - N) * 32; idx += 256) {
            const int r = idx >> 5, col = idx & 31, my = r < off ? r : r + N;
            sf[((col >> 1) * G::FFB + my) * 2 + (col & 1)] = 0.f;
        }
        __syncthreads();
        float2 v[R];
#pragma unroll
        for (int n2 = 0; n2 < R; n2++) v[n2] = ex[t + 16 * n2];
        __syncthreads();
        fft_m<R, -1>(v, t, ex, tw);
#pragma unroll
        for (int m = 0; m < R; m++) ex[out_idx<R>(t, m)] = v[out_slot<R>(m)];
        __syncthreads();
        // C_even[ky] = (Z[ky] + conj Z[M-ky]) / 2, C_odd[ky] = (Z[ky] - conj Z[M-ky]) / (2i)
        for (int idx = tid; idx < H * 32; idx += 256) {
            const int ky = idx >> 5, col = idx & 31, px = c0 + col;
            if (px >= N) continue;
            const float2 *zf = sx + (col >> 1) * G::FFB;
            const float2 z = zf[ky], zm = zf[mirror_idx<M>(ky)];
            tmp[((size_t)a * H + ky) * N + px] = (col & 1)
                ? make_float2(0.5f * (z.y + zm.y), -0.5f * (z.x - zm.x))
                : make_float2(0.5f * (z.x + zm.x), 0.5f * (z.y - zm.y));
        }
    }
}

// C -> CAS images: per spectrum row ky in [0, M/2 + 1) the transform along x
// gives the full row F[ky][.]; CAS row ky and (Hermitian) row M - ky are
// written whole.  Grid (row groups of 16, images).
template <int R>
__global__ __launch_bounds__(256) void k_fwd_rows(const float2 *__restrict__ tmp, float *__restrict__ cas,
                                                  int n, int N, float scale, int zeroNyq)
{
    using G = FftGeom<R>;
    constexpr int M = G::M, H = G::H;
    __shared__ float2 sx[16 * G::FFB];
    __shared__ float2 tw[M];
    load_tw<R>(tw);
    const int tid = threadIdx.x, f = tid >> 4, t = tid & 15;
    const int off = (M - N) / 2;
    const int ky = 16 * blockIdx.x + f;
    const bool rowOk = ky <= M / 2;
    float2 *ex = sx + f * G::FFB;
    for (int a = blockIdx.y; a < n; a += gridDim.y) {
        const float2 *crow = tmp + ((size_t)a * H + (rowOk ? ky : 0)) * N;
        float2 v[R];
#pragma unroll
        for (int n2 = 0; n2 < R; n2++) {
            const int px = t + 16 * n2 - off;
            v[n2] = (rowOk && px >= 0 && px < N) ? crow[px] : make_float2(0.f, 0.f);
        }
        __syncthreads();
        fft_m<R, -1>(v, t, ex, tw);
        if (rowOk) {
            float *o = cas + (size_t)a * M * M;
            const bool mirror = ky != 0 && ky != M / 2;
#pragma unroll
            for (int m = 0; m < R; m++) {
                    const int kx = out_idx<R>(t, m);
                    const float2 F = v[out_slot<R>(m)];
                    const float sd = chk(kx + ky);
                    o[ky * M + kx] = (zeroNyq && (kx == 0 || ky == 0)) ? 0.f : (sd * F.x + sd * F.y) * scale;
                    if (mirror) {
                        const int x = mirror_idx<M>(kx);  // CAS[M - ky][x] from conj F[ky][(M - x) % M]
                        const float sm = chk(x + ky);
                        o[(M - ky) * M + x] = (zeroNyq && x == 0) ? 0.f : (sm * F.x - sm * F.y) * scale;
                    }
                }
        }
    }
}

// ---------------------------------------------------------------------------
// The same two-pass image chains (and the volume chains below) for any other
// even M up to 512 whose prime factors are 2, 3, 5, 7, 11 and 13: the
// transforms run in place in LDS as Stockham passes of radix 10, 8, 6, 4, 2,
// 3, 5, 7, 11 or 13.  A pass reads its butterflies into registers,
// synchronises and writes them back in order.  rocFFT's chain costs five or
// six passes over the padded images and, per call, up to 9 batch sizes of two
// launches each.  300 images, there and back, from rocFFT's chain: M = 50
// 93 -> 21 us, 100 154 -> 39, 200 284 -> 90, 300 695 -> 171, 480 1,674 -> 392
// (3.4 TB/s of the bytes); one image 22-45 -> 17-25 us, launches on both sides.
// A volume, there and back: M = 100 72 -> 40 us, 240 354 -> 127, 300 749 -> 212.
// ---------------------------------------------------------------------------
struct GPass {
    FastDiv ns, count;   // product of the radices before; butterflies of a transform (M / radix)
    unsigned radix, tws;  // twiddle stride M / (ns radix)
};
struct GPlan {
    int M, H, C, passes;  // C transforms per workgroup
    FastDiv m, h, c;
    GPass pass[9];  // 2^9 = 512
};

// R-point DFT of v in place, natural order.  The second halves of the
// constants of 3 and 5 keep their rounding out of the result (M = 100, there
// and back: 1.27e-7 and 1.36e-7 against 1.45e-7 and 1.47e-7 without).
template <int R, int S>
__device__ __forceinline__ void dft_any(float2 (&v)[R], const float2 *tw, int M)
{
    if constexpr (R == 2) {
        const float2 a = v[0], b = v[1];
        v[0] = make_float2(a.x + b.x, a.y + b.y);
        v[1] = make_float2(a.x - b.x, a.y - b.y);
    } else if constexpr (R == 3) {
        constexpr float c = 0.866025403784438647f, c2 = (float)(0.866025403784438647 - (double)c);
        const float sg = S > 0 ? 1.f : -1.f;
        const float2 t = make_float2(v[1].x + v[2].x, v[1].y + v[2].y), u = make_float2(v[1].x - v[2].x, v[1].y - v[2].y);
        const float2 e = make_float2(fmaf(-0.5f, t.x, v[0].x), fmaf(-0.5f, t.y, v[0].y));
        const float2 f = make_float2(sg * fmaf(c, u.x, c2 * u.x), sg * fmaf(c, u.y, c2 * u.y));
        v[0] = make_float2(v[0].x + t.x, v[0].y + t.y);
        v[1] = make_float2(e.x - f.y, e.y + f.x);
        v[2] = make_float2(e.x + f.y, e.y - f.x);
    } else if constexpr (R == 4) {
        fft4<S>(v[0], v[1], v[2], v[3]);
    } else if constexpr (R == 8) {
        fft8<S>(v);
    } else if constexpr (R == 6 || R == 10) {
        // 2 and Q are coprime: no twiddles between the two stages
        constexpr int Q = R / 2;
        float2 a[Q], b[Q];
#pragma unroll
        for (int n = 0; n < Q; n++) {
            const float2 x = v[(2 * n) % R], y = v[(Q + 2 * n) % R];
            a[n] = make_float2(x.x + y.x, x.y + y.y);
            b[n] = make_float2(x.x - y.x, x.y - y.y);
        }
        dft_any<Q, S>(a, tw, M);
        dft_any<Q, S>(b, tw, M);
#pragma unroll
        for (int k = 0; k < Q; k++) {
            v[(k * (Q + 1)) % R] = a[k];
            v[(Q + k * (Q + 1)) % R] = b[k];
        }
    } else if constexpr (R == 5) {
        // cos 72 and cos 144 degrees are -1/4 +- sqrt(5)/4
        constexpr float q = 0.559016994374947424f, q2 = (float)(0.559016994374947424 - (double)q);
        constexpr float s1 = 0.951056516295153572f, s12 = (float)(0.951056516295153572 - (double)s1);
        constexpr float s2 = 0.587785252292473129f, s22 = (float)(0.587785252292473129 - (double)s2);
        const float2 t1 = make_float2(v[1].x + v[4].x, v[1].y + v[4].y), t2 = make_float2(v[2].x + v[3].x, v[2].y + v[3].y);
        const float2 t3 = make_float2(v[1].x - v[4].x, v[1].y - v[4].y), t4 = make_float2(v[2].x - v[3].x, v[2].y - v[3].y);
        const float2 m = make_float2(t1.x + t2.x, t1.y + t2.y), d = make_float2(t1.x - t2.x, t1.y - t2.y);
        const float2 a = make_float2(fmaf(-0.25f, m.x, v[0].x), fmaf(-0.25f, m.y, v[0].y));
        const float2 b = make_float2(fmaf(q2, d.x, q * d.x), fmaf(q2, d.y, q * d.y));
        const float sg = S > 0 ? 1.f : -1.f;
        const float2 e1 = make_float2(a.x + b.x, a.y + b.y), e2 = make_float2(a.x - b.x, a.y - b.y);
        const float2 f1 = make_float2(sg * fmaf(s1, t3.x, fmaf(s2, t4.x, fmaf(s12, t3.x, s22 * t4.x))),
                                      sg * fmaf(s1, t3.y, fmaf(s2, t4.y, fmaf(s12, t3.y, s22 * t4.y))));
        const float2 f2 = make_float2(sg * fmaf(s2, t3.x, fmaf(-s1, t4.x, fmaf(s22, t3.x, -s12 * t4.x))),
                                      sg * fmaf(s2, t3.y, fmaf(-s1, t4.y, fmaf(s22, t3.y, -s12 * t4.y))));
        v[0] = make_float2(v[0].x + m.x, v[0].y + m.y);
        v[1] = make_float2(e1.x - f1.y, e1.y + f1.x);
        v[4] = make_float2(e1.x + f1.y, e1.y - f1.x);
        v[2] = make_float2(e2.x - f2.y, e2.y + f2.x);
        v[3] = make_float2(e2.x + f2.y, e2.y - f2.x);
    } else {
        // odd prime: X[k], X[R - k] from the sums and differences of x[n], x[R - n]
        float2 o[R], p[R / 2], m[R / 2];
        o[0] = make_float2(0.f, 0.f);
#pragma unroll
        for (int n = 1; n <= R / 2; n++) {
            p[n - 1] = make_float2(v[n].x + v[R - n].x, v[n].y + v[R - n].y);
            m[n - 1] = make_float2(v[n].x - v[R - n].x, v[n].y - v[R - n].y);
            o[0] = make_float2(o[0].x + p[n - 1].x, o[0].y + p[n - 1].y);
        }
        o[0] = make_float2(v[0].x + o[0].x, v[0].y + o[0].y);
#pragma unroll
        for (int k = 1; k <= R / 2; k++) {
            float2 e = make_float2(0.f, 0.f), d = make_float2(0.f, 0.f);
#pragma unroll
            for (int n = 1; n <= R / 2; n++) {
                const float2 w = tw[(M / R) * ((n * k) % R)];  // (cos, sin), the same for all lanes
                e.x = fmaf(w.x, p[n - 1].x, e.x);
                e.y = fmaf(w.x, p[n - 1].y, e.y);
                d.x = fmaf(w.y, m[n - 1].x, d.x);
                d.y = fmaf(w.y, m[n - 1].y, d.y);
            }
            e = make_float2(v[0].x + e.x, v[0].y + e.y);  // last: a rounding of v[0] less per term
            const float sg = S > 0 ? 1.f : -1.f;
            o[k] = make_float2(fmaf(-sg, d.y, e.x), fmaf(sg, d.x, e.y));
            o[R - k] = make_float2(fmaf(sg, d.y, e.x), fmaf(-sg, d.x, e.y));
        }
#pragma unroll
        for (int k = 0; k < R; k++) v[k] = o[k];
    }
}

// One pass over C transforms of x (pitch M), by 256 threads; barriers inside.
template <int R, int S, int G>
__device__ __forceinline__ void fft_pass(float2 *x, const float2 *tw, const GPass &p, int M, int C)
{
    constexpr int NB = (G + R - 1) / R;  // C M <= 256 G
    float2 v[NB][R];
    int o[NB];
    const unsigned n = p.count.d, total = (unsigned)C * n;
#pragma unroll
    for (int i = 0; i < NB; i++) {
        const unsigned w = threadIdx.x + 256u * i;
        o[i] = -1;
        if (w < total) {
            const unsigned c = p.count(w), b = w - c * n, blk = p.ns(b), j = b - blk * p.ns.d;
            const float2 *in = x + c * (unsigned)M + b;
            v[i][0] = in[0];
#pragma unroll
            for (int q = 1; q < R; q++) {
                const float2 t = tw[j * p.tws * (unsigned)q];
                v[i][q] = cmulw(in[q * n], t.x, S > 0 ? t.y : -t.y);
            }
            dft_any<R, S>(v[i], tw, M);
            o[i] = (int)(c * (unsigned)M + blk * p.ns.d * (unsigned)R + j);
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NB; i++)
        if (o[i] >= 0) {
#pragma unroll
            for (int q = 0; q < R; q++) x[o[i] + q * (int)p.ns.d] = v[i][q];
        }
    __syncthreads();
}

// C transforms of x in place, natural order; the data must be visible (a
// barrier since the stores).
template <int S, int G>
__device__ __forceinline__ void fft_any(float2 *x, const float2 *tw, const GPlan &P, int C)
{
    for (int i = 0; i < P.passes; i++) {
        const GPass &p = P.pass[i];
        switch (p.radix) {
        case 8: fft_pass<8, S, G>(x, tw, p, P.M, C); break;
        case 10: fft_pass<10, S, G>(x, tw, p, P.M, C); break;
        case 6: fft_pass<6, S, G>(x, tw, p, P.M, C); break;
        case 4: fft_pass<4, S, G>(x, tw, p, P.M, C); break;
        case 2: fft_pass<2, S, G>(x, tw, p, P.M, C); break;
        case 3: fft_pass<3, S, G>(x, tw, p, P.M, C); break;
        case 5: fft_pass<5, S, G>(x, tw, p, P.M, C); break;
        case 7: fft_pass<7, S, G>(x, tw, p, P.M, C); break;
        case 11: fft_pass<11, S, G>(x, tw, p, P.M, C); break;
        default: fft_pass<13, S, G>(x, tw, p, P.M, C); break;
        }
    }
}

__device__ __forceinline__ void load_tw_any(float2 *tw, int M)
{
    for (int q = threadIdx.x; q < M; q += 256) {
        // 2q/M = a + r: the rounding of a is made up to first order
        const float a = (float)(2 * q) / (float)M, r = (float)M_PI * (fmaf(-a, (float)M, (float)(2 * q)) / (float)M);
        float sn, cs;
        sincospif(a, &sn, &cs);
        tw[q] = make_float2(fmaf(-r, sn, cs), fmaf(r, cs, sn));
    }
}

// total items of a workgroup through load and then put, U loads of a thread in
// flight; the clamped last item may be put several times (the same value).
template <int U, typename L, typename F>
__device__ __forceinline__ void g_stage(int total, L load, F put)
{
    for (int b = 0; b < total; b += U * 256) {
        decltype(load(0)) v[U];
#pragma unroll
        for (int i = 0; i < U; i++) v[i] = load(min(b + (int)threadIdx.x + 256 * i, total - 1));
#pragma unroll
        for (int i = 0; i < U; i++) put(min(b + (int)threadIdx.x + 256 * i, total - 1), v[i]);
    }
}

// The four image passes, as k_inv_rows, k_inv_cols, k_fwd_cols and k_fwd_rows
// have them.  Grid: (ceil(H / C) or ceil(N / 2C), images).
template <int G>
__global__ __launch_bounds__(256) void g_inv_rows(const float *__restrict__ cas, float2 *__restrict__ tmp, int n, int N, GPlan P)
{
    __shared__ float2 x[256 * G];
    __shared__ float2 tw[512];
    const int M = P.M, H = P.H, C = P.C, off = (M - N) / 2, ky0 = C * (int)blockIdx.x;
    load_tw_any(tw, M);
    for (int a = blockIdx.y; a < n; a += gridDim.y) {
        const float *im = cas + (size_t)a * M * M;
        g_stage<G>(C * M, [&](int e) {
            const int c = (int)P.m(e), kx = e - c * M, ky = min(ky0 + c, H - 1);
            return make_float2(im[ky * M + kx], im[(ky ? M - ky : 0) * M + (kx ? M - kx : 0)]);
        }, [&](int e, float2 v) {
            const int c = (int)P.m(e), kx = e - c * M, ky = min(ky0 + c, H - 1);
            const float sg = chk(kx + ky);
            x[e] = kx != 0 && ky != 0 ? make_float2(sg * (0.5f * (v.x + v.y)), sg * (0.5f * (v.x - v.y)))
                                      : make_float2(0.f, 0.f);
        });
        __syncthreads();
        fft_any<1, G>(x, tw, P, C);
        for (int e = threadIdx.x; e < C * M; e += 256) {
            const int c = (int)P.m(e), px = e - c * M - off, ky = ky0 + c;
            if (ky < H && px >= 0 && px < N) tmp[((size_t)a * H + ky) * N + px] = x[e];
        }
        __syncthreads();
    }
}

template <int G>
__global__ __launch_bounds__(256) void g_inv_cols(const float2 *__restrict__ tmp, float *__restrict__ imgs, int n, int N,
                                                  float scale, GPlan P)
{
    __shared__ float2 x[256 * G];
    __shared__ float2 tw[512];
    const int M = P.M, H = P.H, C = P.C, off = (M - N) / 2, px0 = 2 * C * (int)blockIdx.x;
    load_tw_any(tw, M);
    for (int a = blockIdx.y; a < n; a += gridDim.y) {
        g_stage<G>(C * H, [&](int e) {  // N is even: columns come in pairs
            const int ky = (int)P.c(e), c = e - ky * C, p0 = min(px0 + 2 * c, N - 2);
            const float2 *r = tmp + ((size_t)a * H + ky) * N + p0;
            return make_float4(r[0].x, r[0].y, r[1].x, r[1].y);
        }, [&](int e, float4 v) {
            const int ky = (int)P.c(e), c = e - ky * C;
            x[c * M + ky] = make_float2(v.x - v.w, v.y + v.z);
            if (ky != 0 && ky != M / 2) x[c * M + M - ky] = make_float2(v.x + v.w, v.z - v.y);
        });
        __syncthreads();
        fft_any<1, G>(x, tw, P, C);
        for (int e = threadIdx.x; e < 2 * C * N; e += 256) {
            const int py = (int)P.c(e >> 1), col = e - py * 2 * C, px = px0 + col, my = py + off;
            if (px >= N) continue;
            const float2 z = x[(col >> 1) * M + my];
            imgs[((size_t)a * N + py) * N + px] = chk(px + off + my) * ((col & 1) ? z.y : z.x) * scale;
        }
        __syncthreads();
    }
}

template <int G>
__global__ __launch_bounds__(256) void g_fwd_cols(const float *__restrict__ imgs, float2 *__restrict__ tmp, int n, int N, GPlan P)
{
    __shared__ float2 x[256 * G];
    __shared__ float2 tw[512];
    const int M = P.M, H = P.H, C = P.C, off = (M - N) / 2, px0 = 2 * C * (int)blockIdx.x;
    load_tw_any(tw, M);
    float *xs = reinterpret_cast<float *>(x);
    for (int a = blockIdx.y; a < n; a += gridDim.y) {
        g_stage<G>(2 * C * M, [&](int e) {
            const int my = (int)P.c(e >> 1), col = e - my * 2 * C, px = px0 + col, py = my - off;
            return imgs[((size_t)a * N + min(max(py, 0), N - 1)) * N + min(px, N - 1)];
        }, [&](int e, float raw) {
            const int my = (int)P.c(e >> 1), col = e - my * 2 * C, px = px0 + col, py = my - off;
            const bool in = py >= 0 && py < N && px < N;
            xs[((col >> 1) * M + my) * 2 + (col & 1)] = in ? chk(px + off + my) * raw : 0.f;
        });
        __syncthreads();
        fft_any<-1, G>(x, tw, P, C);
        for (int e = threadIdx.x; e < 2 * C * H; e += 256) {
            const int ky = (int)P.c(e >> 1), col = e - ky * 2 * C, px = px0 + col;
            if (px >= N) continue;
            const float2 z = x[(col >> 1) * M + ky], zm = x[(col >> 1) * M + (ky ? M - ky : 0)];
            tmp[((size_t)a * H + ky) * N + px] = (col & 1) ? make_float2(0.5f * (z.y + zm.y), -0.5f * (z.x - zm.x))
                                                           : make_float2(0.5f * (z.x + zm.x), 0.5f * (z.y - zm.y));
        }
        __syncthreads();
    }
}

template <int G>
__global__ __launch_bounds__(256) void g_fwd_rows(const float2 *__restrict__ tmp, float *__restrict__ cas, int n, int N,
                                                  float scale, int zeroNyq, GPlan P)
{
    __shared__ float2 x[256 * G];
    __shared__ float2 tw[512];
    const int M = P.M, H = P.H, C = P.C, off = (M - N) / 2, ky0 = C * (int)blockIdx.x;
    load_tw_any(tw, M);
    for (int a = blockIdx.y; a < n; a += gridDim.y) {
        g_stage<G>(C * M, [&](int e) {
            const int c = (int)P.m(e), px = e - c * M - off, ky = min(ky0 + c, H - 1);
            return tmp[((size_t)a * H + ky) * N + min(max(px, 0), N - 1)];
        }, [&](int e, float2 raw) {
            const int c = (int)P.m(e), px = e - c * M - off;
            x[e] = px >= 0 && px < N ? raw : make_float2(0.f, 0.f);
        });
        __syncthreads();
        fft_any<-1, G>(x, tw, P, C);
        float *o = cas + (size_t)a * M * M;
        for (int e = threadIdx.x; e < C * M; e += 256) {
            const int c = (int)P.m(e), kx = e - c * M, ky = ky0 + c;
            if (ky >= H) continue;
            const float2 F = x[e], Fm = x[c * M + (kx ? M - kx : 0)];
            const float sd = chk(kx + ky);
            o[ky * M + kx] = (zeroNyq && (kx == 0 || ky == 0)) ? 0.f : (sd * F.x + sd * F.y) * scale;
            if (ky != 0 && ky != M / 2)  // CAS row M - ky from conj F[ky][(M - kx) % M]
                o[(M - ky) * M + kx] = (zeroNyq && kx == 0) ? 0.f : (sd * Fm.x - sd * Fm.y) * scale;
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// Volume chains (utils/CASFromVol_Gridder.m:34-60, utils/volFromCAS_Gridder.m:
// 37-56).  In 3-D the shift identity carries a global sign (-1)^(3M/2).
// ---------------------------------------------------------------------------
__global__ void k_vol_to_real3d(const float *__restrict__ vol, int N, float *__restrict__ real,
                                int M, const float *__restrict__ pc, size_t total)
{
    const int off = (M - N) / 2;
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (size_t)gridDim.x * blockDim.x) {
        const int mx = (int)(e % M);
        const size_t rest = e / M;
        const int my = (int)(rest % M);
        const int mz = (int)(rest / M);
        const int qx = mx - off, qy = my - off, qz = mz - off;
        float v = 0.f;
        if (qx >= 0 && qx < N && qy >= 0 && qy < N && qz >= 0 && qz < N) {
            const double w = (double)pc[mx] * (double)pc[my] * (double)pc[mz];
            v = chk(mx + my + mz) *
                (float)(w * (double)vol[((size_t)qz * N + qy) * N + qx]);
        }
        real[e] = v;
    }
}

__global__ void k_herm3d_to_casvol(const float2 *__restrict__ herm, int M,
                                   float *__restrict__ casVol, int V, int pad, float gsign,
                                   size_t total)
{
    const int H = M / 2 + 1;
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (size_t)gridDim.x * blockDim.x) {
        const int vx = (int)(e % V);
        const size_t rest = e / V;
        const int vy = (int)(rest % V);
        const int vz = (int)(rest / V);
        const int cx = vx - pad, cy = vy - pad, cz = vz - pad;
        float out = 0.f;
        if (cx >= 0 && cx < M && cy >= 0 && cy < M && cz >= 0 && cz < M) {
            float re, im;
            if (cx <= M / 2) {
                const float2 f = herm[((size_t)cz * M + cy) * H + cx];
                re = f.x; im = f.y;
            } else {
                const float2 f = herm[((size_t)((M - cz) % M) * M + (M - cy) % M) * H + (M - cx)];
                re = f.x; im = -f.y;
            }
            const float s = gsign * chk(cx + cy + cz);
            out = s * re + s * im;
        }
        casVol[e] = out;
    }
}

__global__ void k_casvol_to_herm3d(const float *__restrict__ casVol, int V, int pad,
                                   float2 *__restrict__ herm, int M, int zeroNyq, size_t total)
{
    const int H = M / 2 + 1;
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (size_t)gridDim.x * blockDim.x) {
        const int cx = (int)(e % H);
        const size_t rest = e / H;
        const int cy = (int)(rest % M);
        const int cz = (int)(rest / M);
        float2 z = make_float2(0.f, 0.f);
        if (!(zeroNyq && (cx == 0 || cy == 0 || cz == 0))) {
            const float c1 = casVol[((size_t)(cz + pad) * V + (cy + pad)) * V + (cx + pad)];
            const int mx = (M - cx) % M, my = (M - cy) % M, mz = (M - cz) % M;
            const float c2 = casVol[((size_t)(mz + pad) * V + (my + pad)) * V + (mx + pad)];
            const float s = chk(cx + cy + cz);
            z.x = s * (0.5f * (c1 + c2));
            z.y = s * (0.5f * (c1 - c2));
        }
        herm[e] = z;
    }
}

__global__ void k_real3d_to_vol(const float *__restrict__ real, int M, float *__restrict__ vol,
                                int N, const float *__restrict__ pc, double scale, size_t total)
{
    const int off = (M - N) / 2;
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (size_t)gridDim.x * blockDim.x) {
        const int qx = (int)(e % N);
        const size_t rest = e / N;
        const int qy = (int)(rest % N);
        const int qz = (int)(rest / N);
        const int mx = qx + off, my = qy + off, mz = qz + off;
        const double w = (double)pc[mx] * (double)pc[my] * (double)pc[mz] * scale;
        vol[e] = chk(mx + my + mz) * (float)(w * (double)real[((size_t)mz * M + my) * M + mx]);
    }
}

// ---------------------------------------------------------------------------
// Fused volume chains for the image chains' sizes (M = 128, 192, 256, 384 and
// 512): three passes of one-dimensional transforms (fft_m) that neither read
// nor write the padding.  With A = N x N x H and B = N x M x H complex values
// (H = M/2 + 1, kx fastest) the forward chain goes volume -> A (along x, two
// real rows in one complex transform) -> B (along y) -> CAS volume (along z,
// each value written with its Hermitian mirror), the inverse back the same
// way, keeping N of M outputs along z, y and x.  rocFFT's chain makes seven
// passes over M^3 or V^3 values instead.  Along y and z a workgroup takes 16
// neighbouring kx (lanes: kx fastest, so every load and store is a run of 16),
// and workgroups of one (y, z) line of tiles follow each other on one XCD, so
// that partial lines meet in its L2.  Bound by memory: along z at N=256 3.4 TB/s
// (241 us forward, 825 MB) and 3.1 TB/s (inverse) of the 5.1 TB/s of a copy.
// Both directions together: N=128 437 -> 111 us, N=256 3,835 -> 806 us.
// ---------------------------------------------------------------------------
struct VolLine { int line, kx0; bool ok; };
// The workgroup's line (of n) and its first kx; n * tiles workgroups, rounded
// up to 8 lines.
template <int H>
__device__ __forceinline__ VolLine vol_line(int n)
{
    constexpr int T = (H + 15) / 16;
    const int idx = (int)(blockIdx.x >> 3), q = idx / T;
    const int line = q * 8 + (int)(blockIdx.x & 7u);
    return {line, 16 * (idx - q * T), line < n};
}

// Volume -> A.  Grid: 32 rows per workgroup.
template <int R>
__global__ __launch_bounds__(256) void k_vol_fwd_x(const float *__restrict__ vol, int N, float2 *__restrict__ A,
                                                   const float *__restrict__ pc)
{
    using G = FftGeom<R>;
    constexpr int M = G::M, H = G::H;
    __shared__ float2 sx[16 * G::FFB];
    __shared__ float2 tw[M];
    load_tw<R>(tw);
    const int tid = threadIdx.x, f = tid >> 4, t = tid & 15;
    const int off = (M - N) / 2, rows = N * N;
    const int row0 = 32 * (int)blockIdx.x + 2 * f;
    float2 *ex = sx + f * G::FFB;
    float2 v[R];
    {
        const int r0 = min(row0, rows - 1), r1 = min(row0 + 1, rows - 1);
        const int z0 = r0 / N + off, y0 = r0 % N + off, z1 = r1 / N + off, y1 = r1 % N + off;
        const double w0 = (double)pc[y0] * (double)pc[z0], w1 = (double)pc[y1] * (double)pc[z1];
        const float s0 = chk(y0 + z0), s1 = chk(y1 + z1);
        float a[R], b[R];
#pragma unroll
        for (int n2 = 0; n2 < R; n2++) {  // unconditional loads from clamped addresses
            const int q = min(max(t + 16 * n2 - off, 0), N - 1);
            a[n2] = vol[(size_t)r0 * N + q];
            b[n2] = vol[(size_t)r1 * N + q];
        }
#pragma unroll
        for (int n2 = 0; n2 < R; n2++) {
            const int mx = t + 16 * n2, q = mx - off;
            const bool in = q >= 0 && q < N;
            const double px = (double)pc[mx];
            const float sg = chk(mx);
            v[n2] = make_float2(in ? sg * s0 * (float)(px * w0 * (double)a[n2]) : 0.f,
                                in ? sg * s1 * (float)(px * w1 * (double)b[n2]) : 0.f);
        }
    }
    __syncthreads();
    fft_m<R, -1>(v, t, ex, tw);
#pragma unroll
    for (int m = 0; m < R; m++) ex[out_idx<R>(t, m)] = v[out_slot<R>(m)];
    __syncthreads();
    for (int r = tid >> 6; r < 32; r += 4) {
        const int row = 32 * (int)blockIdx.x + r;
        if (row >= rows) break;
        const float2 *zf = sx + (r >> 1) * G::FFB;
        for (int k = tid & 63; k < H; k += 64) {
            const float2 z = zf[k], zm = zf[mirror_idx<M>(k)];
            A[(size_t)row * H + k] = (r & 1) ? make_float2(0.5f * (z.y + zm.y), -0.5f * (z.x - zm.x))
                                             : make_float2(0.5f * (z.x + zm.x), 0.5f * (z.y - zm.y));
        }
    }
}

// A <-> B, lines z (S = -1: N values of y in, M out; S = 1: M in, N out).
template <int R, int S>
__global__ __launch_bounds__(256) void k_vol_y(const float2 *__restrict__ in, float2 *__restrict__ out, int N)
{
    using G = FftGeom<R>;
    constexpr int M = G::M, H = G::H;
    __shared__ float2 sx[16 * G::FFB];
    __shared__ float2 tw[M];
    load_tw<R>(tw);
    const VolLine l = vol_line<H>(N);
    if (!l.ok) return;  // uniform
    const int tid = threadIdx.x, f = tid & 15, t = tid >> 4, kx = l.kx0 + f, off = (M - N) / 2;
    const int nIn = S < 0 ? N : M, oIn = S < 0 ? off : 0, nOut = S < 0 ? M : N, oOut = S < 0 ? 0 : off;
    const float2 *src = in + (size_t)l.line * nIn * H + min(kx, H - 1);
    float2 v[R];
#pragma unroll
    for (int n2 = 0; n2 < R; n2++) v[n2] = src[(size_t)min(max(t + 16 * n2 - oIn, 0), nIn - 1) * H];
#pragma unroll
    for (int n2 = 0; n2 < R; n2++) {
        const int y = t + 16 * n2 - oIn;
        if (y < 0 || y >= nIn) v[n2] = make_float2(0.f, 0.f);
    }
    __syncthreads();
    fft_m<R, S>(v, t, sx + f * G::FFB, tw);
    if (kx < H) {
        float2 *dst = out + (size_t)l.line * nOut * H + kx;
#pragma unroll
        for (int m = 0; m < R; m++) {
            const int y = out_idx<R>(t, m) - oOut;
            if (y >= 0 && y < nOut) dst[(size_t)y * H] = v[out_slot<R>(m)];
        }
    }
}

// B -> CAS volume, lines ky; the padding shell is k_casvol_shell's.
template <int R>
__global__ __launch_bounds__(256) void k_vol_fwd_z(const float2 *__restrict__ B, int N, float *__restrict__ casVol, int V,
                                                   int pad, float gsign)
{
    using G = FftGeom<R>;
    constexpr int M = G::M, H = G::H;
    __shared__ float2 sx[16 * G::FFB];
    __shared__ float2 tw[M];
    load_tw<R>(tw);
    const VolLine l = vol_line<H>(M);
    if (!l.ok) return;  // uniform
    const int tid = threadIdx.x, f = tid & 15, t = tid >> 4, kx = l.kx0 + f, ky = l.line, off = (M - N) / 2;
    const float2 *src = B + (size_t)ky * H + min(kx, H - 1);
    float2 v[R];
#pragma unroll
    for (int n2 = 0; n2 < R; n2++) v[n2] = src[(size_t)min(max(t + 16 * n2 - off, 0), N - 1) * M * H];
#pragma unroll
    for (int n2 = 0; n2 < R; n2++) {
        const int z = t + 16 * n2 - off;
        if (z < 0 || z >= N) v[n2] = make_float2(0.f, 0.f);
    }
    __syncthreads();
    fft_m<R, -1>(v, t, sx + f * G::FFB, tw);
    if (kx >= H) return;
    const bool mirror = kx != 0 && kx != M / 2;
    const int my = mirror_idx<M>(ky);
#pragma unroll
    for (int m = 0; m < R; m++) {
        const int kz = out_idx<R>(t, m);
        const float2 F = v[out_slot<R>(m)];
        const float s = gsign * chk(kx + ky + kz);  // the mirror's indices have the same parity
        casVol[((size_t)(kz + pad) * V + (ky + pad)) * V + (kx + pad)] = s * F.x + s * F.y;
        if (mirror)
            casVol[((size_t)(mirror_idx<M>(kz) + pad) * V + (my + pad)) * V + (M - kx + pad)] = s * F.x - s * F.y;
    }
}

// The CAS volume's padding: rows outside the M x M centre whole, the others'
// ends.  Grid (V planes, 8), a row per wave.
__global__ __launch_bounds__(256) void k_casvol_shell(float *__restrict__ casVol, int V, int pad)
{
    const int z = (int)blockIdx.x, ln = threadIdx.x & 63;
    for (int y = (int)blockIdx.y * 4 + (int)(threadIdx.x >> 6); y < V; y += (int)gridDim.y * 4) {
        float *row = casVol + ((size_t)z * V + y) * V;
        const bool inside = y >= pad && y < V - pad && z >= pad && z < V - pad;
        for (int x = ln; x < (inside ? 2 * pad : V); x += 64) row[inside && x >= pad ? V - 2 * pad + x : x] = 0.f;
    }
}

// CAS volume -> B, lines ky.
template <int R>
__global__ __launch_bounds__(256) void k_vol_inv_z(const float *__restrict__ casVol, int V, int pad,
                                                   float2 *__restrict__ B, int N, int zeroNyq)
{
    using G = FftGeom<R>;
    constexpr int M = G::M, H = G::H;
    __shared__ float2 sx[16 * G::FFB];
    __shared__ float2 tw[M];
    load_tw<R>(tw);
    const VolLine l = vol_line<H>(M);
    if (!l.ok) return;  // uniform
    const int tid = threadIdx.x, f = tid & 15, t = tid >> 4, kx = l.kx0 + f, ky = l.line, off = (M - N) / 2;
    const int xs = min(kx, H - 1), my = mirror_idx<M>(ky), mx = mirror_idx<M>(xs);
    const float *p1 = casVol + ((size_t)pad * V + (ky + pad)) * V + (xs + pad);
    const float *p2 = casVol + ((size_t)pad * V + (my + pad)) * V + (mx + pad);
    const size_t VV = (size_t)V * V;
    float c1[R], c2[R];
#pragma unroll
    for (int n2 = 0; n2 < R; n2++) {
        const int kz = t + 16 * n2;
        c1[n2] = p1[kz * VV];
        c2[n2] = p2[mirror_idx<M>(kz) * VV];
    }
    float2 v[R];
#pragma unroll
    for (int n2 = 0; n2 < R; n2++) {
        const int kz = t + 16 * n2;
        const float s = chk(kx + ky + kz);
        const bool drop = zeroNyq && (kx == 0 || ky == 0 || kz == 0);  // whatever is there, NaN included
        v[n2] = drop ? make_float2(0.f, 0.f)
                     : make_float2(s * (0.5f * (c1[n2] + c2[n2])), s * (0.5f * (c1[n2] - c2[n2])));
    }
    __syncthreads();
    fft_m<R, 1>(v, t, sx + f * G::FFB, tw);
    if (kx >= H) return;
    float2 *dst = B + (size_t)ky * H + kx;
#pragma unroll
    for (int m = 0; m < R; m++) {
        const int z = out_idx<R>(t, m) - off;
        if (z >= 0 && z < N) dst[(size_t)z * M * H] = v[out_slot<R>(m)];
    }
}

// A -> volume: two Hermitian rows per complex transform, whose real and
// imaginary outputs are the two real rows.  Grid: 32 rows per workgroup.
template <int R>
__global__ __launch_bounds__(256) void k_vol_inv_x(const float2 *__restrict__ A, float *__restrict__ vol, int N,
                                                   const float *__restrict__ pc, double scale)
{
    using G = FftGeom<R>;
    constexpr int M = G::M, H = G::H;
    __shared__ float2 sx[16 * G::FFB];
    __shared__ float2 tw[M];
    load_tw<R>(tw);
    const int tid = threadIdx.x, f = tid >> 4, t = tid & 15;
    const int off = (M - N) / 2, rows = N * N;
    const int row0 = 32 * (int)blockIdx.x + 2 * f;
    const int r0 = min(row0, rows - 1), r1 = min(row0 + 1, rows - 1);
    const float2 *a0 = A + (size_t)r0 * H, *a1 = A + (size_t)r1 * H;
    float2 v[R];
#pragma unroll
    for (int n2 = 0; n2 < R; n2++) {
        const int k = t + 16 * n2;
        const bool up = k > M / 2;
        const float2 p = a0[up ? M - k : k], q = a1[up ? M - k : k];
        v[n2] = up ? make_float2(p.x + q.y, q.x - p.y) : make_float2(p.x - q.y, p.y + q.x);
        // a real transform has no imaginary part at k = 0 and M/2
        if (k == 0 || k == M / 2) v[n2] = make_float2(p.x, q.x);
    }
    __syncthreads();
    fft_m<R, 1>(v, t, sx + f * G::FFB, tw);
    const int z0 = r0 / N + off, y0 = r0 % N + off, z1 = r1 / N + off, y1 = r1 % N + off;
    const double w0 = (double)pc[y0] * (double)pc[z0] * scale, w1 = (double)pc[y1] * (double)pc[z1] * scale;
    const float s0 = chk(y0 + z0), s1 = chk(y1 + z1);
#pragma unroll
    for (int m = 0; m < R; m++) {
        const int mx = out_idx<R>(t, m), px = mx - off;
        if (px < 0 || px >= N) continue;
        const float2 z = v[out_slot<R>(m)];
        const double w = (double)pc[mx];
        const float sg = chk(mx);
        if (row0 < rows) vol[(size_t)row0 * N + px] = sg * s0 * (float)(w * w0 * (double)z.x);
        if (row0 + 1 < rows) vol[(size_t)(row0 + 1) * N + px] = sg * s1 * (float)(w * w1 * (double)z.y);
    }
}

// The volume passes for the other sizes (fft_any).  Along y and z a workgroup
// takes C neighbouring kx of one line.
__device__ __forceinline__ VolLine g_vol_line(int n, int tiles, int C)
{
    const int idx = (int)(blockIdx.x >> 3), q = idx / tiles;
    const int line = q * 8 + (int)(blockIdx.x & 7u);
    return {line, C * (idx - q * tiles), line < n};
}

template <int G>
__global__ __launch_bounds__(256) void g_vol_fwd_x(const float *__restrict__ vol, int N, float2 *__restrict__ A,
                                                   const float *__restrict__ pc, GPlan P)
{
    __shared__ float2 x[256 * G];
    __shared__ float2 tw[512];
    const int M = P.M, H = P.H, C = P.C, off = (M - N) / 2, rows = N * N, row0 = 2 * C * (int)blockIdx.x;
    load_tw_any(tw, M);
    float *xs = reinterpret_cast<float *>(x);
    g_stage<G>(2 * C * M, [&](int e) {
        const int r = (int)P.m(e), mx = e - r * M, row = min(row0 + r, rows - 1);
        return vol[(size_t)row * N + min(max(mx - off, 0), N - 1)];
    }, [&](int e, float raw) {
        const int r = (int)P.m(e), mx = e - r * M, q = mx - off, row = min(row0 + r, rows - 1);
        const int mz = row / N + off, my = row % N + off;
        const double w = (double)pc[mx] * (double)pc[my] * (double)pc[mz];
        xs[((r >> 1) * M + mx) * 2 + (r & 1)] = q >= 0 && q < N ? chk(mx + my + mz) * (float)(w * (double)raw) : 0.f;
    });
    __syncthreads();
    fft_any<-1, G>(x, tw, P, C);
    for (int e = threadIdx.x; e < 2 * C * H; e += 256) {
        const int r = (int)P.h(e), k = e - r * H, row = row0 + r;
        if (row >= rows) break;
        const float2 z = x[(r >> 1) * M + k], zm = x[(r >> 1) * M + (k ? M - k : 0)];
        A[(size_t)row * H + k] = (r & 1) ? make_float2(0.5f * (z.y + zm.y), -0.5f * (z.x - zm.x))
                                         : make_float2(0.5f * (z.x + zm.x), 0.5f * (z.y - zm.y));
    }
}

template <int S, int G>
__global__ __launch_bounds__(256) void g_vol_y(const float2 *__restrict__ in, float2 *__restrict__ out, int N, int tiles, GPlan P)
{
    __shared__ float2 x[256 * G];
    __shared__ float2 tw[512];
    const int M = P.M, H = P.H, C = P.C, off = (M - N) / 2;
    load_tw_any(tw, M);
    const VolLine l = g_vol_line(N, tiles, C);
    if (!l.ok) return;  // uniform
    const int nIn = S < 0 ? N : M, oIn = S < 0 ? off : 0, nOut = S < 0 ? M : N, oOut = S < 0 ? 0 : off;
    g_stage<G>(C * M, [&](int e) {
        const int my = (int)P.c(e), c = e - my * C, y = my - oIn;
        return in[((size_t)l.line * nIn + min(max(y, 0), nIn - 1)) * H + min(l.kx0 + c, H - 1)];
    }, [&](int e, float2 raw) {
        const int my = (int)P.c(e), c = e - my * C, y = my - oIn;
        x[c * M + my] = y >= 0 && y < nIn ? raw : make_float2(0.f, 0.f);
    });
    __syncthreads();
    fft_any<S, G>(x, tw, P, C);
    for (int e = threadIdx.x; e < C * nOut; e += 256) {
        const int y = (int)P.c(e), c = e - y * C;
        if (l.kx0 + c < H) out[((size_t)l.line * nOut + y) * H + l.kx0 + c] = x[c * M + y + oOut];
    }
}

template <int G>
__global__ __launch_bounds__(256) void g_vol_fwd_z(const float2 *__restrict__ B, int N, float *__restrict__ casVol, int V,
                                                   int pad, float gsign, int tiles, GPlan P)
{
    __shared__ float2 x[256 * G];
    __shared__ float2 tw[512];
    const int M = P.M, H = P.H, C = P.C, off = (M - N) / 2;
    load_tw_any(tw, M);
    const VolLine l = g_vol_line(M, tiles, C);
    if (!l.ok) return;  // uniform
    const int ky = l.line, my = ky ? M - ky : 0;
    g_stage<G>(C * M, [&](int e) {
        const int mz = (int)P.c(e), c = e - mz * C, z = mz - off;
        return B[((size_t)min(max(z, 0), N - 1) * M + ky) * H + min(l.kx0 + c, H - 1)];
    }, [&](int e, float2 raw) {
        const int mz = (int)P.c(e), c = e - mz * C, z = mz - off;
        x[c * M + mz] = z >= 0 && z < N ? raw : make_float2(0.f, 0.f);
    });
    __syncthreads();
    fft_any<-1, G>(x, tw, P, C);
    for (int e = threadIdx.x; e < C * M; e += 256) {
        const int kz = (int)P.c(e), c = e - kz * C, kx = l.kx0 + c;
        if (kx >= H) continue;
        const float2 F = x[c * M + kz];
        const float s = gsign * chk(kx + ky + kz);
        casVol[((size_t)(kz + pad) * V + (ky + pad)) * V + (kx + pad)] = s * F.x + s * F.y;
        if (kx != 0 && kx != M / 2)
            casVol[((size_t)((kz ? M - kz : 0) + pad) * V + (my + pad)) * V + (M - kx + pad)] = s * F.x - s * F.y;
    }
}

template <int G>
__global__ __launch_bounds__(256) void g_vol_inv_z(const float *__restrict__ casVol, int V, int pad, float2 *__restrict__ B,
                                                   int N, int zeroNyq, int tiles, GPlan P)
{
    __shared__ float2 x[256 * G];
    __shared__ float2 tw[512];
    const int M = P.M, H = P.H, C = P.C, off = (M - N) / 2;
    load_tw_any(tw, M);
    const VolLine l = g_vol_line(M, tiles, C);
    if (!l.ok) return;  // uniform
    const int ky = l.line, my = ky ? M - ky : 0;
    g_stage<G>(C * M, [&](int e) {
        const int kz = (int)P.c(e), c = e - kz * C, kx = min(l.kx0 + c, H - 1);
        return make_float2(casVol[((size_t)(kz + pad) * V + (ky + pad)) * V + (kx + pad)],
                           casVol[((size_t)((kz ? M - kz : 0) + pad) * V + (my + pad)) * V + ((kx ? M - kx : 0) + pad)]);
    }, [&](int e, float2 v) {
        const int kz = (int)P.c(e), c = e - kz * C, kx = min(l.kx0 + c, H - 1);
        const float c1 = v.x, c2 = v.y, s = chk(kx + ky + kz);
        const bool drop = zeroNyq && (kx == 0 || ky == 0 || kz == 0);  // whatever is there, NaN included
        x[c * M + kz] = drop ? make_float2(0.f, 0.f) : make_float2(s * (0.5f * (c1 + c2)), s * (0.5f * (c1 - c2)));
    });
    __syncthreads();
    fft_any<1, G>(x, tw, P, C);
    for (int e = threadIdx.x; e < C * N; e += 256) {
        const int z = (int)P.c(e), c = e - z * C;
        if (l.kx0 + c < H) B[((size_t)z * M + ky) * H + l.kx0 + c] = x[c * M + z + off];
    }
}

template <int G>
__global__ __launch_bounds__(256) void g_vol_inv_x(const float2 *__restrict__ A, float *__restrict__ vol, int N,
                                                   const float *__restrict__ pc, double scale, GPlan P)
{
    __shared__ float2 x[256 * G];
    __shared__ float2 tw[512];
    const int M = P.M, H = P.H, C = P.C, off = (M - N) / 2, rows = N * N, row0 = 2 * C * (int)blockIdx.x;
    load_tw_any(tw, M);
    g_stage<G>(C * H, [&](int e) {
        const int c = (int)P.h(e), k = e - c * H;
        const float2 p = A[(size_t)min(row0 + 2 * c, rows - 1) * H + k], q = A[(size_t)min(row0 + 2 * c + 1, rows - 1) * H + k];
        return make_float4(p.x, p.y, q.x, q.y);
    }, [&](int e, float4 v) {
        const int c = (int)P.h(e), k = e - c * H;
        const float2 p = make_float2(v.x, v.y), q = make_float2(v.z, v.w);
        // a real transform has no imaginary part at k = 0 and M/2
        const bool real = k == 0 || k == M / 2;
        x[c * M + k] = real ? make_float2(p.x, q.x) : make_float2(p.x - q.y, p.y + q.x);
        if (!real) x[c * M + M - k] = make_float2(p.x + q.y, q.x - p.y);
    });
    __syncthreads();
    fft_any<1, G>(x, tw, P, C);
    for (int e = threadIdx.x; e < 2 * C * M; e += 256) {
        const int r = (int)P.m(e), mx = e - r * M, px = mx - off, row = row0 + r;
        if (px < 0 || px >= N || row >= rows) continue;
        const int mz = row / N + off, my = row % N + off;
        const float2 z = x[(r >> 1) * M + mx];
        const double w = (double)pc[mx] * (double)pc[my] * (double)pc[mz] * scale;
        vol[(size_t)row * N + px] = chk(mx + my + mz) * (float)(w * (double)((r & 1) ? z.y : z.x));
    }
}

// ---------------------------------------------------------------------------
// Reductions, conversions, fills.
// ---------------------------------------------------------------------------
__global__ void k_reduce_partials(float *__restrict__ out, const float *__restrict__ parts,
                                  int nParts, size_t n, size_t stride, int accumulate)
{
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
         e += (size_t)gridDim.x * blockDim.x) {
        double s = accumulate ? (double)out[e] : 0.0;
        for (int q = 0; q < nParts; q++) s += (double)parts[(size_t)q * stride + e];
        out[e] = (float)s;
    }
}

__global__ void k_divide_density(float *__restrict__ out, const float *__restrict__ num,
                                 const float *__restrict__ den, size_t n, double eps)
{
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
         e += (size_t)gridDim.x * blockDim.x)
        out[e] = (float)((double)num[e] / ((double)den[e] + eps));
}

__global__ void k_to_bf16(uint16_t *__restrict__ dst, const float *__restrict__ src, size_t n)
{
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
         e += (size_t)gridDim.x * blockDim.x) {
        uint32_t u = __float_as_uint(src[e]);
        if ((u & 0x7f800000u) == 0x7f800000u) {  // inf / nan: truncate, keep nan quiet
            dst[e] = (uint16_t)((u >> 16) | ((u & 0x007fffffu) ? 0x40u : 0u));
        } else {
            u += 0x7fffu + ((u >> 16) & 1u);  // round to nearest even
            dst[e] = (uint16_t)(u >> 16);
        }
    }
}

__global__ void k_to_f16(uint16_t *__restrict__ dst, const float *__restrict__ src, size_t n)
{
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
         e += (size_t)gridDim.x * blockDim.x) {
        __half h = __float2half_rn(src[e]);
        dst[e] = __half_raw(h).x;
    }
}

__global__ void k_fill(float *__restrict__ p, float v, size_t n)
{
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
         e += (size_t)gridDim.x * blockDim.x)
        p[e] = v;
}

// ---------------------------------------------------------------------------
// Check behind the forward projector's 4-wide windows: *check = 1 when the
// table has the 501 entries, all finite, with both end entries 0, and every
// value of the volume is finite; else 0.  k_check_table (one workgroup) writes
// the table's verdict, then k_check_volume clears it on any non-finite voxel
// (all finding workgroups store the same 0).
// ---------------------------------------------------------------------------
__global__ void k_check_table(const float *__restrict__ ker, int K, unsigned *__restrict__ check, unsigned good)
{
    bool ok = true;
    for (int t = threadIdx.x; t < K; t += blockDim.x) ok = ok && __builtin_isfinite(ker[t]);
    ok = __syncthreads_and(ok);
    if (threadIdx.x == 0) *check = (ok && K == KFP_FAST && ker[0] == 0.f && ker[K - 1] == 0.f) ? good : 0u;
}

// Non-finite = exponent field all ones (FP32 0x7f800000, BF16 0x7f80, FP16 0x7c00).
// The calling thread's share of n FP32 values.
__device__ __forceinline__ bool any_nonfinite(const unsigned *__restrict__ w, size_t n)
{
    const size_t t0 = (size_t)blockIdx.x * blockDim.x + threadIdx.x, st = (size_t)gridDim.x * blockDim.x;
    bool bad = false;
    size_t e0 = 0;
    if (((uintptr_t)w & 15u) == 0) {  // 16-byte loads over the aligned body
        const size_t n4 = n / 4;
        const u4 *w4 = (const u4 *)w;
        for (size_t e = t0; e < n4; e += st) {
            const u4 q = w4[e];
            bad |= ((q.x & 0x7f800000u) == 0x7f800000u) | ((q.y & 0x7f800000u) == 0x7f800000u) |
                   ((q.z & 0x7f800000u) == 0x7f800000u) | ((q.w & 0x7f800000u) == 0x7f800000u);
        }
        e0 = n4 * 4;
    }
    for (size_t e = e0 + t0; e < n; e += st) bad |= (w[e] & 0x7f800000u) == 0x7f800000u;
    return bad;
}

template <int DT>
__global__ void k_check_volume(const void *__restrict__ vol, size_t n, unsigned *__restrict__ check)
{
    bool bad = false;
    if (DT == DT_F32) {
        bad = any_nonfinite((const unsigned *)vol, n);
    } else {
        const size_t t0 = (size_t)blockIdx.x * blockDim.x + threadIdx.x, st = (size_t)gridDim.x * blockDim.x;
        const uint16_t *h = (const uint16_t *)vol;
        const unsigned m = DT == DT_BF16 ? 0x7f80u : 0x7c00u;
        for (size_t e = t0; e < n; e += st) bad |= ((unsigned)h[e] & m) == m;
    }
    if (__syncthreads_or(bad) && threadIdx.x == 0) *check = 0u;
}

// *check = 3 where another flag says that table and images are finite.
__global__ void k_check_from(const unsigned *__restrict__ finite, unsigned *__restrict__ check)
{
    *check = *finite == 1u ? 3u : 0u;
}

// The check behind the column kernels: k_check_table has set *check
// to 3 or 0; a non-finite image value clears both bits (everything is left to
// the other kernel), a frame that is not orthonormal to tol the second (that
// frame is; planes: only [u v] counts).
__global__ void k_check_back(const float *__restrict__ img, size_t n, const float *__restrict__ axes, int nAxes,
                             float tol, int planes, unsigned *__restrict__ check)
{
    const bool bad = any_nonfinite((const unsigned *)img, n);
    bool skew = false;
    for (int a = blockIdx.x * blockDim.x + threadIdx.x; a < nAxes; a += gridDim.x * blockDim.x) {
        float a9[9];
#pragma unroll
        for (int k = 0; k < 9; k++) a9[k] = axes[(size_t)9 * a + k];
        skew = skew || !(planes ? adj_plane(a9, tol) : bp_orthonormal(a9, tol));
    }
    const bool anyBad = __syncthreads_or(bad), anySkew = __syncthreads_or(skew);
    if (threadIdx.x == 0) {
        if (anyBad) atomicAnd(check, 0u);
        else if (anySkew) atomicAnd(check, 1u);
    }
}

// ---------------------------------------------------------------------------
// Standalone filters (Filters/*.cu).  Same element semantics as the reference
// kernels; grid-stride 1-D launches instead of one thread per (x, y) column.
// ---------------------------------------------------------------------------
__global__ void k_f_cas_to_complex(const float *__restrict__ in, float2 *__restrict__ out, int S,
                                   int nSlices, int volumeMode, size_t total)
{
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (size_t)gridDim.x * blockDim.x) {
        const int i = (int)(e % S);
        const size_t rest = e / S;
        const int j = (int)(rest % S);
        const int k = (int)(rest / S);
        float2 z = make_float2(0.f, 0.f);
        const bool skip = volumeMode ? (i == 0 || j == 0 || k == 0) : (i == 0 || j == 0);
        if (!skip) {
            const int k2 = volumeMode ? S - k : k;
            const size_t n2 = (size_t)(S - i) + (size_t)(S - j) * S + (size_t)k2 * S * S;
            z.x = 0.5f * (in[e] + in[n2]);
            z.y = 0.5f * (in[e] - in[n2]);
        }
        out[e] = z;
    }
}

__global__ void k_f_complex_to_cas(const float2 *__restrict__ in, float *__restrict__ out, size_t n)
{
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
         e += (size_t)gridDim.x * blockDim.x)
        out[e] = in[e].x + in[e].y;
}

__global__ void k_f_complex_to_real(const float2 *__restrict__ in, float *__restrict__ out, size_t n)
{
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
         e += (size_t)gridDim.x * blockDim.x)
        out[e] = in[e].x;
}

__global__ void k_f_real_to_complex(const float *__restrict__ in, float2 *__restrict__ out, size_t n)
{
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
         e += (size_t)gridDim.x * blockDim.x)
        out[e] = make_float2(in[e], 0.f);
}

// In-place quadrant swap per slice (even S): element (x, y) with y < S/2
// swaps with ((x + S/2) mod S, y + S/2).
template <typename T>
__global__ void k_f_fftshift2d(T *__restrict__ d, int S, size_t total)
{
    const int h = S / 2;
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (size_t)gridDim.x * blockDim.x) {
        const int x = (int)(e % S);
        const size_t rest = e / S;
        const int y = (int)(rest % h);
        const size_t k = rest / h;
        const size_t a = k * S * S + (size_t)y * S + x;
        const size_t b = k * S * S + (size_t)(y + h) * S + ((x + h) % S);
        T t = d[a];
        d[a] = d[b];
        d[b] = t;
    }
}

// In-place octant swap (even S): element (x, y, z) with z < S/2 swaps with
// ((x + S/2) mod S, (y + S/2) mod S, z + S/2).
template <typename T>
__global__ void k_f_fftshift3d(T *__restrict__ d, int S, size_t total)
{
    const int h = S / 2;
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (size_t)gridDim.x * blockDim.x) {
        const int x = (int)(e % S);
        const size_t rest = e / S;
        const int y = (int)(rest % S);
        const int z = (int)(rest / S);
        const size_t a = ((size_t)z * S + y) * S + x;
        const size_t b = ((size_t)(z + h) * S + (y + h) % S) * S + (x + h) % S;
        T t = d[a];
        d[a] = d[b];
        d[b] = t;
    }
}

__global__ void k_f_pad(const float *__restrict__ in, float *__restrict__ out, int inS, int outS,
                        size_t total)
{
    const int off = (outS - inS) / 2;
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (size_t)gridDim.x * blockDim.x) {
        const int x = (int)(e % outS);
        const size_t rest = e / outS;
        const int y = (int)(rest % outS);
        const size_t k = rest / outS;
        const int ix = x - off, iy = y - off;
        float v = 0.f;
        if (ix >= 0 && ix < inS && iy >= 0 && iy < inS) v = in[k * inS * inS + (size_t)iy * inS + ix];
        out[e] = v;
    }
}

template <typename T>
__global__ void k_f_crop(const T *__restrict__ in, T *__restrict__ out, int inS, int outS,
                         size_t total)
{
    const int off = (inS - outS) / 2;
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (size_t)gridDim.x * blockDim.x) {
        const int x = (int)(e % outS);
        const size_t rest = e / outS;
        const int y = (int)(rest % outS);
        const size_t k = rest / outS;
        out[e] = in[k * inS * inS + (size_t)(y + off) * inS + (x + off)];
    }
}

__global__ void k_f_divide_scalar(float *__restrict__ d, float s, size_t n)
{
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
         e += (size_t)gridDim.x * blockDim.x)
        d[e] = d[e] / s;
}

__global__ void k_f_divide_volume(float *__restrict__ a, const float *__restrict__ b, size_t n)
{
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
         e += (size_t)gridDim.x * blockDim.x) {
        const float x = a[e], y = b[e];
        a[e] = (x != 0.f && y != 0.f) ? x / y : 0.f;
    }
}

__global__ void k_f_multiply_volume(float *__restrict__ a, const float *__restrict__ b, size_t n)
{
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
         e += (size_t)gridDim.x * blockDim.x)
        a[e] = a[e] * b[e];
}

__global__ void k_f_multiply_complex_volume(float2 *__restrict__ a, const float *__restrict__ b,
                                            size_t n)
{
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
         e += (size_t)gridDim.x * blockDim.x) {
        float2 z = a[e];
        z.x = z.x * b[e];
        z.y = z.y * b[e];
        a[e] = z;
    }
}

__global__ void k_f_add_volume(float *__restrict__ a, const float *__restrict__ b, size_t n)
{
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
         e += (size_t)gridDim.x * blockDim.x)
        a[e] = a[e] + b[e];
}

// 1-D grid-stride launch geometry: enough blocks to fill 256 CUs many times
// over, capped so huge arrays loop inside the kernel.
inline unsigned grid_for(size_t n)
{
    size_t g = (n + kThreads - 1) / kThreads;
    if (g > 65536) g = 65536;
    if (g == 0) g = 1;
    return (unsigned)g;
}

// Largest integer d2 (a squared voxel distance, at most 3*(v/2)^2) with
// sqrtf((float)d2) <= r, i.e. the integer form of the reference's mask test
// sqrtf(...) <= maskRadius (gpuBackProject.cu:48-50).  -1 if none passes.
inline int mask_d2(float r, int v)
{
    const long long hi = 3LL * (v / 2 + 1) * (v / 2 + 1);
    if (!(sqrtf(0.f) <= r)) return -1;
    long long lo = 0, top = hi;  // sqrtf is monotone: binary search the last passing d2
    if (sqrtf((float)top) <= r) return (int)top;
    while (top - lo > 1) {
        const long long mid = (lo + top) / 2;
        if (sqrtf((float)mid) <= r) lo = mid; else top = mid;
    }
    return (int)lo;
}

// The mask radius as the reference's kernels see it: RunKernel takes it as an
// int (gpuForwardProject.h:57, gpuBackProject.h:56) from the float member
// (gpuGridder.cpp:262,422), so it is truncated toward zero.  NaN and values
// beyond the int range (no meaningful conversion) pass through.
inline float ref_mask_radius(float r)
{
    if (!(r > -2147483648.0f && r < 2147483648.0f)) return r;
    return (float)(int)r;
}

inline void proj_consts(const ProjGeom &g, float &kerScale, float &kerCenter, float &fW,
                        int &convW)
{
    // gpuForwardProject.cu:20-23: kerCenter = (K-1)/2, kerScale = kerCenter/kerHWidth.
    kerCenter = ((float)g.K - 1) / 2;
    kerScale = kerCenter / g.kerHWidth;
    convW = (int)roundf(g.kerHWidth);
    fW = (float)convW;
}

}  // namespace

// ===========================================================================
// Launchers
// ===========================================================================
hipError_t launch_forward_project(const void *vol, int dtype, const ProjGeom &g,
                                  const float *axes, int nAxes, float *casImgs, hipStream_t s,
                                  const unsigned *check)
{
    if (nAxes <= 0) return hipSuccess;
    FPArgs a;
    a.vol = vol; a.axes = axes; a.out = casImgs; a.ker = g.ker; a.check = nullptr;
    a.columns = nullptr; a.orthTol = 0.f;
    a.V = g.V; a.M = g.M; a.K = g.K; a.nAxes = nAxes;
    a.maskR = ref_mask_radius(g.maskRadius);
    proj_consts(g, a.kerScale, a.kerCenter, a.fW, a.convW);
    const bool w2 = a.convW == 2 && g.K <= FPKER;
    if (w2) {
        // LDS-staged kernel: 8x8 tiles, one per wave, 4 per workgroup.
        const bool fast = a.kerScale == 125.0f && a.kerCenter == 250.0f && g.K == 501;
        a.check = fast ? check : nullptr;
        a.tilesPerRow = (g.M + FPT - 1) / FPT;
        a.tilesPerImg = a.tilesPerRow * a.tilesPerRow;
        a.maskD2 = mask_d2(a.maskR, g.V);
        const unsigned long long work = (unsigned long long)a.tilesPerImg * nAxes;
        if (work > 0xffffffffull / 2) return hipErrorInvalidValue;
        a.totalWork = (unsigned)work;
        a.perXcd = 0;
        // Units of whole images from 256 directions on, where the XCDs' shares
        // even out; bands below (64 directions at N=256: 328 us against 337 by
        // whole images, 5-wide windows 502 against 529).
        FPWalk &wk = a.walk;
        const unsigned cols = (unsigned)(a.tilesPerRow + 1) / 2;
        unsigned bands = 1;
        while (bands < 8 && bands < cols && (unsigned)nAxes * bands < 256u) bands *= 2;
        wk.rows = cols;
        wk.bandRows = (cols + bands - 1) / bands;
        wk.cols.set(cols);
        wk.bands.set(bands);
        wk.unitTiles.set(cols * wk.bandRows);
        wk.units = (unsigned)nAxes * bands;
        wk.perXcd = (wk.units + 7) / 8 * cols * wk.bandRows;
        // A band meets the mask's disc more or less by its place in the image,
        // so each XCD takes every place in turn (16 directions at N=256: 88 ->
        // 85 us, 5-wide windows 146 -> 137).
        wk.turn = bands > 1 ? 7u : 0u;
        // Tiles per wave, a stride of the grid apart: the most that do not
        // leave the last round of the card's 1,024 resident workgroups short,
        // by the cost of 1 / 2 / 3 / 4 of them in a long launch (2,000 random
        // directions at N=128: 2.33 / 2.13 / 2.07 / 2.07 ms; without a check,
        // and so a phase table, 64 at N=256: 530 / 531 / 542 / 548 us).  16
        // directions at N=96, 2,304 workgroup tiles: 17.3 / 19.4 / 16.8 / 19.6
        // us; 2 at N=64, unchecked: 11.5 / 13.5 / 19.4 / 24.8 us.
        const double checked[5] = {0.0, 1.12, 1.03, 1.0, 1.0}, unchecked[5] = {0.0, 1.03, 1.0, 1.02, 1.02};
        const double *weight = a.check ? checked : unchecked;
        const double tiles = 8.0 * wk.perXcd;
        unsigned tpw = 4;
        double least = 0.0;
        for (unsigned k = 4; k >= 1; k--) {
            const double cost = std::ceil(tiles / (1024.0 * k)) * k * weight[k];
            if (k == 4 || cost < least) least = cost, tpw = k;
        }
        const dim3 grid((wk.perXcd + tpw - 1) / tpw * 8), block(kThreads);
        // volumes of 4 GB and more: box addressing from the box's first element
        const int esz = dtype == DT_F32 ? 4 : 2;
        const bool big = (long long)g.V * g.V * g.V * esz >= (1LL << 32);
#define MGG_FP_LAUNCH(DTV)                                                                   \
    if (big) {                                                                               \
        if (fast) hipLaunchKernelGGL((fp_lds_kernel<DTV, true, true>), grid, block, 0, s, a);  \
        else hipLaunchKernelGGL((fp_lds_kernel<DTV, false, true>), grid, block, 0, s, a);      \
    } else if (fast) hipLaunchKernelGGL((fp_lds_kernel<DTV, true, false>), grid, block, 0, s, a); \
    else hipLaunchKernelGGL((fp_lds_kernel<DTV, false, false>), grid, block, 0, s, a);
        switch (dtype) {
        case DT_F32: MGG_FP_LAUNCH(DT_F32) break;
        case DT_BF16: MGG_FP_LAUNCH(DT_BF16) break;
        case DT_F16: MGG_FP_LAUNCH(DT_F16) break;
        default: return hipErrorInvalidValue;
        }
#undef MGG_FP_LAUNCH
        return hipGetLastError();
    }
    a.tilesPerRow = (g.M + 15) / 16;
    a.tilesPerImg = a.tilesPerRow * a.tilesPerRow;
    const unsigned long long work = (unsigned long long)a.tilesPerImg * nAxes;
    if (work > 0xffffffffull / 2) return hipErrorInvalidValue;
    a.totalWork = (unsigned)work;
    a.perXcd = (a.totalWork + 7) / 8;
    const dim3 grid(a.perXcd * 8), block(kThreads);
    const bool rows = a.convW == 2;  // 5-tap row loads (tables too large for the staged kernel)
    switch (dtype) {
    case DT_F32:
        if (rows) hipLaunchKernelGGL((fp_kernel<DT_F32, true>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((fp_kernel<DT_F32, false>), grid, block, 0, s, a);
        break;
    case DT_BF16:
        if (rows) hipLaunchKernelGGL((fp_kernel<DT_BF16, true>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((fp_kernel<DT_BF16, false>), grid, block, 0, s, a);
        break;
    case DT_F16:
        if (rows) hipLaunchKernelGGL((fp_kernel<DT_F16, true>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((fp_kernel<DT_F16, false>), grid, block, 0, s, a);
        break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

bool fp_segment_supported(const ProjGeom &g)
{
    float kerScale, kerCenter, fW;
    int convW;
    proj_consts(g, kerScale, kerCenter, fW, convW);
    return convW == 2 && kerScale == 125.0f && kerCenter == 250.0f && g.K == KFP_FAST && g.K <= FPKER;
}

unsigned fp_segment(FPSegment &sg, const void *vol, const ProjGeom &g, const float *axes, int nAxes, float *casImgs,
                    unsigned workStart, const unsigned *check)
{
    sg.vol = vol; sg.axes = axes; sg.out = casImgs; sg.ker = g.ker; sg.check = check;
    sg.V = g.V; sg.M = g.M; sg.nAxes = nAxes;
    sg.maskD2 = mask_d2(ref_mask_radius(g.maskRadius), g.V);
    sg.tilesPerRow = (g.M + FPT - 1) / FPT;
    sg.tilesPerImg = sg.tilesPerRow * sg.tilesPerRow;
    sg.workStart = workStart;
    return (unsigned)sg.tilesPerImg * (unsigned)nAxes;
}

hipError_t launch_forward_project_multi(const FPMultiArgs &m, hipStream_t s)
{
    if (m.nSegs <= 0 || m.totalWork == 0) return hipSuccess;
    if (m.nSegs > kFpMaxSegments) return hipErrorInvalidValue;
    // The single-volume launch's grid: three tiles per wave, a grid-stride
    // apart.  A persistent grid (no more workgroups than are resident, each
    // walking the list) ran 25% slower on the same tiles.
    const unsigned grid = (m.totalWork + 11) / 12;
    bool big = false;  // a volume of 4 GB or more
    for (int i = 0; i < m.nSegs; i++) big |= (long long)m.seg[i].V * m.seg[i].V * m.seg[i].V * 4 >= (1LL << 32);
    if (big) hipLaunchKernelGGL((fp_lds_multi_kernel<DT_F32, true>), dim3(grid), dim3(kThreads), 0, s, m);
    else hipLaunchKernelGGL((fp_lds_multi_kernel<DT_F32, false>), dim3(grid), dim3(kThreads), 0, s, m);
    return hipGetLastError();
}

bool bp_uses_fast_path(const ProjGeom &g)
{
    float kerScale, kerCenter, fW;
    int convW;
    proj_consts(g, kerScale, kerCenter, fW, convW);
    return convW == 2 && kerScale == 125.0f && kerCenter == 250.0f && g.K == KFAST && g.V <= 8192;
}

int bp_brick_count(int V, int depth)
{
    const int b = (V + BB - 1) / BB;
    return b * b * ((V + depth - 1) / depth);
}

void bp_brick_order(int V, int depth, int *out)
{
    // Bricks of BB x BB x depth sorted by the distance of their centre from
    // the volume centre (ties by index): central bricks, which every
    // direction's slab crosses, are dispatched first.
    const int nb = (V + BB - 1) / BB, nz = (V + depth - 1) / depth;
    const double c = V / 2;
    struct Item { double d; int id; };
    std::vector<Item> items;
    items.reserve((size_t)nb * nb * nz);
    for (int z = 0; z < nz; z++)
        for (int y = 0; y < nb; y++)
            for (int x = 0; x < nb; x++) {
                const double dx = x * BB + 0.5 * (BB - 1) - c, dy = y * BB + 0.5 * (BB - 1) - c,
                             dz = z * depth + 0.5 * (depth - 1) - c;
                items.push_back({dx * dx + dy * dy + dz * dz, (z * nb + y) * nb + x});
            }
    std::sort(items.begin(), items.end(),
              [](const Item &a, const Item &b) { return a.d < b.d || (a.d == b.d && a.id < b.id); });
    for (size_t i = 0; i < items.size(); i++) out[i] = items[i].id;
}

static BPArgs bp_args(float *volAcc, float *densAcc, const ProjGeom &g, const float *axes, int nAxes, const float *casImgs)
{
    BPArgs a;
    a.vol = volAcc; a.dens = densAcc; a.axes = axes; a.img = casImgs; a.ker = g.ker;
    a.V = g.V; a.M = g.M; a.K = g.K; a.nAxes = nAxes;
    a.maskR = ref_mask_radius(g.maskRadius); a.hw = g.kerHWidth;
    proj_consts(g, a.kerScale, a.kerCenter, a.fW, a.convW);
    a.maskD2 = mask_d2(a.maskR, g.V);
    {
        int r = 0;  // floor(sqrt(maskD2))
        while ((long long)(r + 1) * (r + 1) <= (long long)a.maskD2) r++;
        a.maskLo = a.maskD2 < 0 ? g.V : g.V / 2 - r;
    }
    // In-mask voxel: |v - c| <= maskR; orthonormal frame (to 1e-4): |u|, |v| <=
    // 1.00005, and the FP32 evaluation of fi adds < 1e-3.  Then fi, fj >=
    // M/2 - 1.00005 maskR - 1e-3, which must be >= 0.5 for floor(fi + 0.5) to be
    // roundf(fi) (for 0.25 <= x < 0.5 an FP32 x + 0.5 can round up to 1).
    a.posRound = ((double)(g.M / 2) - 1.00005 * (double)a.maskR - 1e-3 >= 0.5) ? 1 : 0;
    // The column kernel's pixel lists and slab bounds allow 5e-3 of error in
    // where the frame puts a voxel of the mask's radius.
    a.orthTol = (float)std::min(1e-4, 2e-3 / std::max(1.0, (double)a.maskR));
    a.check = nullptr;
    a.order = nullptr;
    a.perXcd = a.totalWork = 0;
    return a;
}

hipError_t launch_back_project_adjoint(float *volAcc, const ProjGeom &g, const float *axes,
                                       int nAxes, const float *casImgs, hipStream_t s, const unsigned *check,
                                       const unsigned *columns)
{
    if (nAxes <= 0) return hipSuccess;
    FPArgs a;
    a.vol = nullptr; a.axes = axes; a.out = nullptr; a.ker = g.ker; a.check = nullptr;
    a.columns = columns;
    a.orthTol = bp_args(nullptr, nullptr, g, axes, nAxes, nullptr).orthTol;
    a.V = g.V; a.M = g.M; a.K = g.K; a.nAxes = nAxes;
    a.maskR = ref_mask_radius(g.maskRadius);
    proj_consts(g, a.kerScale, a.kerCenter, a.fW, a.convW);
    if (a.convW == 2 && g.K <= FPKER) {
        // LDS-box scatter: 8x8 tiles, one per wave, 4 per workgroup.
        const bool fast = a.kerScale == 125.0f && a.kerCenter == 250.0f && g.K == 501;
        a.check = fast ? check : nullptr;
        a.tilesPerRow = (g.M + FPT - 1) / FPT;
        a.tilesPerImg = a.tilesPerRow * a.tilesPerRow;
        a.maskD2 = mask_d2(a.maskR, g.V);
        const unsigned long long work = (unsigned long long)a.tilesPerImg * nAxes;
        if (work > 0xffffffffull / 2) return hipErrorInvalidValue;
        a.totalWork = (unsigned)work;
        a.perXcd = 0;
        // one tile per wave; after the column launches usually nothing is left
        const unsigned tiles = (a.totalWork + 3) / 4;
        const dim3 grid(columns ? std::min(tiles, 8192u) : tiles), block(kThreads);
        if (fast) hipLaunchKernelGGL(adj_lds_kernel<true>, grid, block, 0, s, a, casImgs, volAcc);
        else hipLaunchKernelGGL(adj_lds_kernel<false>, grid, block, 0, s, a, casImgs, volAcc);
        return hipGetLastError();
    }
    a.tilesPerRow = (g.M + 15) / 16;
    a.tilesPerImg = a.tilesPerRow * a.tilesPerRow;
    const unsigned long long work = (unsigned long long)a.tilesPerImg * nAxes;
    if (work > 0xffffffffull / 2) return hipErrorInvalidValue;
    a.totalWork = (unsigned)work;
    a.perXcd = (a.totalWork + 7) / 8;
    hipLaunchKernelGGL(adj_kernel, dim3(a.perXcd * 8), dim3(kThreads), 0, s, a, casImgs, volAcc);
    return hipGetLastError();
}

// Distance of the volume's centre from the nearest face of the bricks of 8: 0
// (the centre is on a face, or the voxel before one), 1, or 2 and more.  With the
// centre well inside a brick that brick meets every direction and sets the
// time; on a corner eight share them (4 waves, 1,000 directions: N=92 1.90 ms,
// N=96 2.94).
static int centre_depth(int V)
{
    const int c = V / 2 % 8;
    return std::min(c, 7 - c);
}

// Where the column kernels win (they cost more per block, the bricks by their
// central one, the tiles' atomics more per direction).  Time by columns over
// the time by the better number of waves per brick, random directions:
//   centre depth 0  N=60: 256 1.42, 500 1.21, 1,000 1.06; N=76: 1.33, 1.14, 0.96; N=92: 1.28, 1.11, 0.98;
//     N=100: 1.45, 1.27, 1.11, 1,500 1.04; N=116: 1.30, 1.16, 1.03, 1.00; N=124: 1.28, 1.15, 1.02, 0.99
//   1  N=62: 256 1.30, 500 1.11, 1,000 0.94; N=86: 1.10, 1.06, 0.93; N=102: 1.25, 1.07, 0.92; N=110: 1.33, 1.20, 1.04
//   2, 3  N=32: 256 0.59; N=64: 256 1.12, 500 0.94; N=80: 500 1.04, 1,000 0.87; N=88: 256 1.04, 500 1.00; N=96: 256 0.93;
//     N=104: 256 1.04, 500 0.91; N=112: 256 1.11, 500 0.99; N=120: 500 1.13, 1,000 0.97; N=128: 1,000 0.98
//   N=140: 700 1.00, 1,000 0.96; N=160: 500 1.03; N=192: 500 0.98; N=256: 500 0.94
// The transpose over the tiles: N=80 1,000 0.99; N=96: 500 1.02, 700 0.94; N=108: 500 0.95; N=112: 256 1.05, 500 0.96;
//   N=120: 256 1.04, 500 0.94; N=124: 256 1.00; N=128: 256 0.91; N=146: 256 1.00; N=160: 350 0.98, 500 0.91
bool uses_columns(const ProjGeom &g, int nAxes, ColKind kind)
{
    const bool adjoint = kind == ColKind::Adjoint;
    const int depth = centre_depth(g.V);
    const int least = adjoint ? (g.V < 190 ? INT_MAX : g.V < 230 ? 800 : g.V < 250 ? 500 : g.V < 300 ? 256 : 500)
                      : g.V >= 300 ? 500
                      : g.V >= 240 ? 1000
                      : depth == 0 ? 1500
                      : depth == 1 ? 800
                      : g.V < 110 || (g.V >= 180 && g.V < 220) ? 256 : 500;
    if (nAxes < least || !bp_uses_fast_path(g)) return false;
    const BPArgs a = bp_args(nullptr, nullptr, g, nullptr, nAxes, nullptr);
    if (a.maskD2 < 0) return false;
    // The transpose's windows stay inside the volume (no wrap of the linear
    // index) and its pixels inside the image.
    if (adjoint)
        return a.maskLo >= BP_FORM_A_MIN + 1 && (long long)a.maskD2 <= (long long)(g.M / 2 - 1) * (g.M / 2 - 1);
    return a.posRound && a.maskLo >= BP_FORM_A_MIN;
}

// Waves per brick of bp_fast_kernel.  A small volume's bricks do not fill the
// GPU, and the central ones set the time: eight waves halve it (the density the
// same).  Elsewhere the passes' leftover groups of more waves cost more.  Time
// with eight waves over four: N=38 1 direction 0.98, 8 0.75; N=48 1 1.08, 16
// 0.70; N=64 16 1.21, 32 0.80; N=68 32 1.14, 64 0.85; N=72 32 1.09, 64 0.74;
// N=77 64 1.09, 128 0.90; N=80 128 0.68; N=84 128 1.09 (centre depth 0), N=88
// 0.84, N=90 0.96 (2, 3); N=100 256 1.50; N=104 256 1.15.
static int bp_fast_waves(int V, int nAxes)
{
    const int least = V <= 82 ? 0 : V <= 110 ? 16 : V <= 140 ? 32 : V <= 150 ? 64
                      : V <= 172 || (V <= 190 && centre_depth(V) >= 2) ? 128 : INT_MAX;
    return nAxes >= least ? 8 : 4;
}

int col_depth(ColKind kind) { return bc_depth((int)kind); }

hipError_t launch_check_back(const float *casImgs, const ProjGeom &g, const float *axes, int nAxes, bool planes,
                             unsigned *check, hipStream_t s, const unsigned *finite)
{
    const BPArgs a = bp_args(nullptr, nullptr, g, axes, nAxes, casImgs);
    const size_t n = finite ? 0 : (size_t)std::max(nAxes, 0) * g.M * g.M;
    if (finite) hipLaunchKernelGGL(k_check_from, dim3(1), dim3(1), 0, s, finite, check);
    else hipLaunchKernelGGL(k_check_table, dim3(1), dim3(kThreads), 0, s, g.ker, g.K, check, 3u);
    if (nAxes <= 0) return hipGetLastError();
    const unsigned grid = std::min(grid_for(std::max(n, (size_t)nAxes)), 4096u);
    hipLaunchKernelGGL(k_check_back, dim3(grid), dim3(kThreads), 0, s, casImgs, n, axes, nAxes, a.orthTol, planes ? 1 : 0,
                       check);
    return hipGetLastError();
}

template <int MODE, int W>
static void col_launches(const BPColArgs &a, unsigned blocks, hipStream_t s)
{
    hipLaunchKernelGGL((col_kernel<2, MODE, W>), dim3(blocks), dim3(64 * W), 0, s, a);
    hipLaunchKernelGGL((col_kernel<1, MODE, W>), dim3(blocks), dim3(64 * W), 0, s, a);
    hipLaunchKernelGGL((col_kernel<0, MODE, W>), dim3(blocks), dim3(64 * W), 0, s, a);
}

hipError_t launch_columns(ColKind kind, float *volAcc, const ProjGeom &g, const float *axes, int nAxes,
                          const float *casImgs, hipStream_t s, const int *order, int orderLen, const unsigned *check)
{
    if (nAxes <= 0) return hipSuccess;
    if (!uses_columns(g, nAxes, kind) || !check || !order ||
        orderLen != bp_brick_count(g.V, col_depth(kind)))
        return hipErrorInvalidValue;
    BPColArgs a;
    a.b = bp_args(volAcc, nullptr, g, axes, nAxes, casImgs);
    a.b.check = check;
    a.b.order = order;
    a.blocks8 = (g.V + BCN - 1) / BCN;
    a.reachD2 = a.b.maskD2;
    if (kind == ColKind::Adjoint) {
        // pixels are within sqrt(maskD2) (times the frame's tolerance) of the
        // centre, their voxels less than 2 further along each axis
        const double r = std::sqrt((double)std::max(a.b.maskD2, 0)) * (1.0 + 1e-4) + 3.5;
        a.reachD2 = (int)std::ceil(r * r);
    }
    // Small volumes have few blocks, and the central ones' chain of directions
    // sets the time: eight waves share it (time over four waves': N=64, 500
    // directions 0.68; N=80 0.87; N=84 0.94; N=92 1.11; N=96, 256 1.20).
    if (kind == ColKind::Adjoint) col_launches<COL_ADJOINT, 4>(a, (unsigned)orderLen, s);
    else if (g.V <= 176) col_launches<COL_BACK, 8>(a, (unsigned)orderLen, s);
    else col_launches<COL_BACK, 4>(a, (unsigned)orderLen, s);
    return hipGetLastError();
}

hipError_t launch_back_project(float *volAcc, float *densAcc, const ProjGeom &g,
                               const float *axes, int nAxes, const float *casImgs, hipStream_t s,
                               const int *brickOrder, int orderLen, const unsigned *check)
{
    if (nAxes <= 0) return hipSuccess;
    BPArgs a = bp_args(volAcc, densAcc, g, axes, nAxes, casImgs);
    const bool fast = bp_uses_fast_path(g);
    const int ex = fast ? BB : BPX, ey = fast ? BB : BPY, ez = fast ? BB : BPZ;
    a.bricksX = (g.V + ex - 1) / ex;
    const int bricksY = (g.V + ey - 1) / ey;
    const int bricksZ = (g.V + ez - 1) / ez;
    a.bricksXY = a.bricksX * bricksY;
    a.totalWork = (unsigned)a.bricksXY * (unsigned)bricksZ;
    a.perXcd = (a.totalWork + 7) / 8;
    a.order = brickOrder;
    a.check = check;
    const dim3 grid(a.perXcd * 8), block(kThreads);
    if (fast) {
        if (!brickOrder || orderLen != (int)a.totalWork) return hipErrorInvalidValue;
        const dim3 g1(a.totalWork);
        if (bp_fast_waves(g.V, nAxes) == 8) {
            if (densAcc) hipLaunchKernelGGL((bp_fast_kernel<true, 8>), g1, dim3(512), 0, s, a);
            else hipLaunchKernelGGL((bp_fast_kernel<false, 8>), g1, dim3(512), 0, s, a);
        } else if (densAcc) hipLaunchKernelGGL((bp_fast_kernel<true, 4>), g1, block, 0, s, a);
        else hipLaunchKernelGGL((bp_fast_kernel<false, 4>), g1, block, 0, s, a);
    } else {
        if (check) return hipErrorInvalidValue;
        if (densAcc) hipLaunchKernelGGL(bp_kernel<true>, grid, block, 0, s, a);
        else hipLaunchKernelGGL(bp_kernel<false>, grid, block, 0, s, a);
    }
    return hipGetLastError();
}

// Threads per row workgroup of the 2-D chain kernels: the row length rounded
// up to a wave, at most 256 (longer rows loop).
static int row_threads(int len) { return std::min(256, std::max(64, (len + 63) / 64 * 64)); }
static dim3 rows_grid(int rows, int n) { return dim3((unsigned)rows, (unsigned)std::min(n, 65535)); }

hipError_t launch_cas_to_herm2d(const float *cas, float2 *herm, int M, int n, hipStream_t s)
{
    if (n <= 0 || M <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_cas_to_herm2d, rows_grid(M, n), dim3(row_threads(M / 2 + 1)), 0, s, cas, herm, M, n);
    return hipGetLastError();
}

hipError_t launch_real2d_to_imgs(const float *real, float *imgs, int M, int N, int n, float scale,
                                 hipStream_t s)
{
    if (n <= 0 || N <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_real2d_to_imgs, rows_grid(N, n), dim3(row_threads(N)), 0, s, real, imgs, M, N, scale, n);
    return hipGetLastError();
}

hipError_t launch_imgs_to_real2d(const float *imgs, float *real, int M, int N, int n, hipStream_t s)
{
    if (n <= 0 || M <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_imgs_to_real2d, rows_grid(M, n), dim3(row_threads(M)), 0, s, imgs, real, M, N, n);
    return hipGetLastError();
}

hipError_t launch_herm2d_to_cas(const float2 *herm, float *cas, int M, int n, hipStream_t s, float scale,
                                int zeroNyq)
{
    if (n <= 0 || M <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_herm2d_to_cas, rows_grid(M, n), dim3(row_threads(M)), 0, s, herm, cas, M, n, scale,
                       zeroNyq);
    return hipGetLastError();
}

bool fused_chain_supported(int M, int N)
{
    return (M == 128 || M == 192 || M == 256 || M == 384 || M == 512) && N >= 1 && N <= M;
}

// Radices of M for fft_any; false when M has a prime factor beyond 13, is odd
// or does not fit.  Factors 2 that do not make up an 8 go with a 5 or a 3.
static bool g_plan(int M, GPlan &P)
{
    if (M < 2 || M % 2 || M > 512) return false;
    P.M = M;
    P.H = M / 2 + 1;
    P.m.set((unsigned)M);
    P.h.set((unsigned)P.H);
    P.passes = 0;
    int left = M;
    unsigned ns = 1;
    const auto take = [&](unsigned r) {
        GPass &p = P.pass[P.passes++];
        p.radix = r;
        p.ns.set(ns);
        p.count.set((unsigned)M / r);
        ns *= r;
        p.tws = (unsigned)M / ns;
        left /= (int)r;
    };
    const auto twos = [&] {
        int n = 0;
        while (left % (2 << n) == 0) n++;
        return n % 3;
    };
    for (unsigned r : {10u, 6u})
        while (left % (int)r == 0 && twos()) take(r);
    for (unsigned r : {8u, 4u, 2u, 3u, 5u, 7u, 11u, 13u})
        while (left % (int)r == 0) take(r);
    return left == 1;
}

// Values a thread holds in fft_any (G) and the transforms of a workgroup (C M
// <= 256 G, at most 16) for n lines, reps times.  The kernels are as long as G
// and a short launch waits for its instructions: 4 while 8 would leave the
// card with less than four workgroups per CU (one image of M = 240: 17.9 us
// with 16, 13.2 with 4; 300 images of M = 200: 58 with 16, 48 with 8; of M =
// 480: 218 with 8, 282 with 4).
static int g_split(GPlan &P, int n, size_t reps, unsigned &groups)
{
    int most = 0, G = 8;
    for (;; G = 4) {
        most = std::min(16, 256 * G / P.M);
        if (G == 4 || (size_t)((n + most - 1) / most) * reps >= 1024) break;
    }
    const int even = (n + most - 1) / most;
    P.C = (n + even - 1) / even;
    P.c.set((unsigned)P.C);
    groups = (unsigned)((n + P.C - 1) / P.C);
    return G;
}
#define MGG_G(G, kernel, kernel8, ...)                              \
    do {                                                            \
        if ((G) == 4) hipLaunchKernelGGL((kernel), __VA_ARGS__);    \
        else hipLaunchKernelGGL((kernel8), __VA_ARGS__);            \
    } while (0)

// Whether an image chain takes k_inv_rows and its like.  Their threads hold M /
// 16 values and the lines beside the cropped images cost them as much as any:
// at M = 384 and 512 the general passes are faster up to about N = 5/8 M (M =
// 512, there and back: N = 256 300 images 473 -> 423 us, 16 61 -> 53, one 40 ->
// 25; N = 512 300 images 758 against 790; M = 384: N = 192 16 images 39.9
// against 39.2, N = 288 44.7 against 46.4).
static bool own_image_passes(int M, int N) { return fused_chain_supported(M, N) && (M < 384 || 8 * N > 5 * M); }

bool image_chain_supported(int M, int N)
{
    GPlan P;
    return N >= 1 && N <= M && (fused_chain_supported(M, N) || ((M - N) % 2 == 0 && g_plan(M, P)));  // N even
}

template <int R>
static void fused_inverse(const float *cas, float2 *tmp, float *imgs, int N, int n, float scale, hipStream_t s)
{
    constexpr int H = 8 * R + 1;
    const unsigned ny = (unsigned)std::min(n, 65535);
    hipLaunchKernelGGL(k_inv_rows<R>, dim3((H + 15) / 16, ny), dim3(256), 0, s, cas, tmp, n, N);
    hipLaunchKernelGGL(k_inv_cols<R>, dim3((unsigned)((N + 31) / 32), ny), dim3(256), 0, s, tmp, imgs, n, N,
                       scale);
}

template <int R>
static void fused_forward(const float *imgs, float2 *tmp, float *cas, int N, int n, float scale, int zeroNyq,
                          hipStream_t s)
{
    constexpr int H = 8 * R + 1;
    const unsigned ny = (unsigned)std::min(n, 65535);
    hipLaunchKernelGGL(k_fwd_cols<R>, dim3((unsigned)((N + 31) / 32), ny), dim3(256), 0, s, imgs, tmp, n, N);
    hipLaunchKernelGGL(k_fwd_rows<R>, dim3((H + 15) / 16, ny), dim3(256), 0, s, tmp, cas, n, N, scale, zeroNyq);
}

hipError_t launch_fused_cas_to_images(const float *cas, float2 *tmp, float *imgs, int M, int N, int n,
                                      float scale, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    if (!image_chain_supported(M, N)) return hipErrorInvalidValue;
    if (!own_image_passes(M, N)) {
        GPlan P;
        if (!g_plan(M, P)) return hipErrorInvalidValue;
        const unsigned ny = (unsigned)std::min(n, 65535);
        unsigned groups = 0;
        int G = g_split(P, P.H, (size_t)n, groups);
        MGG_G(G, (g_inv_rows<4>), (g_inv_rows<8>), dim3(groups, ny), dim3(256), 0, s, cas, tmp, n, N, P);
        G = g_split(P, N / 2, (size_t)n, groups);
        MGG_G(G, (g_inv_cols<4>), (g_inv_cols<8>), dim3(groups, ny), dim3(256), 0, s, tmp, imgs, n, N, scale, P);
        return hipGetLastError();
    }
    switch (M) {
    case 128: fused_inverse<8>(cas, tmp, imgs, N, n, scale, s); break;
    case 192: fused_inverse<12>(cas, tmp, imgs, N, n, scale, s); break;
    case 256: fused_inverse<16>(cas, tmp, imgs, N, n, scale, s); break;
    case 384: fused_inverse<24>(cas, tmp, imgs, N, n, scale, s); break;
    default: fused_inverse<32>(cas, tmp, imgs, N, n, scale, s); break;
    }
    return hipGetLastError();
}

hipError_t launch_fused_images_to_cas(const float *imgs, float2 *tmp, float *cas, int M, int N, int n,
                                      float scale, int zeroNyq, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    if (!image_chain_supported(M, N)) return hipErrorInvalidValue;
    if (!own_image_passes(M, N)) {
        GPlan P;
        if (!g_plan(M, P)) return hipErrorInvalidValue;
        const unsigned ny = (unsigned)std::min(n, 65535);
        unsigned groups = 0;
        int G = g_split(P, N / 2, (size_t)n, groups);
        MGG_G(G, (g_fwd_cols<4>), (g_fwd_cols<8>), dim3(groups, ny), dim3(256), 0, s, imgs, tmp, n, N, P);
        G = g_split(P, P.H, (size_t)n, groups);
        MGG_G(G, (g_fwd_rows<4>), (g_fwd_rows<8>), dim3(groups, ny), dim3(256), 0, s, tmp, cas, n, N, scale, zeroNyq, P);
        return hipGetLastError();
    }
    switch (M) {
    case 128: fused_forward<8>(imgs, tmp, cas, N, n, scale, zeroNyq, s); break;
    case 192: fused_forward<12>(imgs, tmp, cas, N, n, scale, zeroNyq, s); break;
    case 256: fused_forward<16>(imgs, tmp, cas, N, n, scale, zeroNyq, s); break;
    case 384: fused_forward<24>(imgs, tmp, cas, N, n, scale, zeroNyq, s); break;
    default: fused_forward<32>(imgs, tmp, cas, N, n, scale, zeroNyq, s); break;
    }
    return hipGetLastError();
}

bool fused_volume_supported(int M, int N)
{
    // B (N M H complex) has to fit the M^3 real scratch
    // Below M = 80 one rocFFT plan's few launches are as fast or faster than
    // the general passes (M = 64: 17 us against 18; 80: 42 against 39 there and
    // back; 100: 71 against 41).
    return image_chain_supported(M, N) && M >= 80 && N % 2 == 0 && (size_t)N * (M + 2) <= (size_t)M * M;
}

template <int R>
static void fused_vol_fwd(const float *vol, int N, float *casVol, int V, int pad, const float *pc, float2 *A, float2 *B,
                          float gsign, hipStream_t s)
{
    constexpr int M = 16 * R, T = (M / 2 + 1 + 15) / 16;
    const unsigned rows = (unsigned)((N * N + 31) / 32);
    hipLaunchKernelGGL(k_vol_fwd_x<R>, dim3(rows), dim3(256), 0, s, vol, N, A, pc);
    hipLaunchKernelGGL((k_vol_y<R, -1>), dim3((unsigned)((N + 7) / 8 * 8 * T)), dim3(256), 0, s, A, B, N);
    if (pad > 0)
        hipLaunchKernelGGL(k_casvol_shell, dim3((unsigned)V, 8), dim3(256), 0, s, casVol, V, pad);
    hipLaunchKernelGGL(k_vol_fwd_z<R>, dim3((unsigned)(M * T)), dim3(256), 0, s, B, N, casVol, V, pad, gsign);
}

template <int R>
static void fused_vol_inv(const float *casVol, int V, int pad, float *vol, int N, const float *pc, float2 *A, float2 *B,
                          int zeroNyq, double scale, hipStream_t s)
{
    constexpr int M = 16 * R, T = (M / 2 + 1 + 15) / 16;
    hipLaunchKernelGGL(k_vol_inv_z<R>, dim3((unsigned)(M * T)), dim3(256), 0, s, casVol, V, pad, B, N, zeroNyq);
    hipLaunchKernelGGL((k_vol_y<R, 1>), dim3((unsigned)((N + 7) / 8 * 8 * T)), dim3(256), 0, s, B, A, N);
    hipLaunchKernelGGL(k_vol_inv_x<R>, dim3((unsigned)((N * N + 31) / 32)), dim3(256), 0, s, A, vol, N, pc, scale);
}

hipError_t launch_fused_volume_to_cas(const float *vol, int N, float *casVol, int M, int pad, const float *precomp,
                                      float2 *a, float2 *b, hipStream_t s)
{
    if (!fused_volume_supported(M, N)) return hipErrorInvalidValue;
    const float g = ((3 * (M / 2)) & 1) ? -1.f : 1.f;
    const int V = M + 2 * pad;
    if (!fused_chain_supported(M, N)) {
        GPlan P;
        if (!g_plan(M, P)) return hipErrorInvalidValue;
        unsigned T = 0;
        int G = g_split(P, N * N / 2, 1, T);
        MGG_G(G, (g_vol_fwd_x<4>), (g_vol_fwd_x<8>), dim3(T), dim3(256), 0, s, vol, N, a, precomp, P);
        G = g_split(P, P.H, (size_t)N, T);
        MGG_G(G, (g_vol_y<-1, 4>), (g_vol_y<-1, 8>), dim3((unsigned)(N + 7) / 8 * 8 * T), dim3(256), 0, s, a, b, N,
              (int)T, P);
        if (pad > 0) hipLaunchKernelGGL(k_casvol_shell, dim3((unsigned)V, 8), dim3(256), 0, s, casVol, V, pad);
        G = g_split(P, P.H, (size_t)M, T);
        MGG_G(G, (g_vol_fwd_z<4>), (g_vol_fwd_z<8>), dim3((unsigned)(M + 7) / 8 * 8 * T), dim3(256), 0, s, b, N, casVol, V,
              pad, g, (int)T, P);
        return hipGetLastError();
    }
    switch (M) {
    case 128: fused_vol_fwd<8>(vol, N, casVol, V, pad, precomp, a, b, g, s); break;
    case 192: fused_vol_fwd<12>(vol, N, casVol, V, pad, precomp, a, b, g, s); break;
    case 256: fused_vol_fwd<16>(vol, N, casVol, V, pad, precomp, a, b, g, s); break;
    case 384: fused_vol_fwd<24>(vol, N, casVol, V, pad, precomp, a, b, g, s); break;
    default: fused_vol_fwd<32>(vol, N, casVol, V, pad, precomp, a, b, g, s); break;
    }
    return hipGetLastError();
}

hipError_t launch_fused_cas_to_volume(const float *casVol, int M, int pad, float *vol, int N, const float *precomp,
                                      int zeroNyquist, float scale, float2 *a, float2 *b, hipStream_t s)
{
    if (!fused_volume_supported(M, N)) return hipErrorInvalidValue;
    const double sc = (((3 * (M / 2)) & 1) ? -1.0 : 1.0) * (double)scale;
    const int V = M + 2 * pad;
    if (!fused_chain_supported(M, N)) {
        GPlan P;
        if (!g_plan(M, P)) return hipErrorInvalidValue;
        unsigned T = 0;
        int G = g_split(P, P.H, (size_t)M, T);
        MGG_G(G, (g_vol_inv_z<4>), (g_vol_inv_z<8>), dim3((unsigned)(M + 7) / 8 * 8 * T), dim3(256), 0, s, casVol, V, pad, b, N,
              zeroNyquist, (int)T, P);
        G = g_split(P, P.H, (size_t)N, T);
        MGG_G(G, (g_vol_y<1, 4>), (g_vol_y<1, 8>), dim3((unsigned)(N + 7) / 8 * 8 * T), dim3(256), 0, s, b, a, N,
              (int)T, P);
        G = g_split(P, N * N / 2, 1, T);
        MGG_G(G, (g_vol_inv_x<4>), (g_vol_inv_x<8>), dim3(T), dim3(256), 0, s, a, vol, N, precomp, sc, P);
        return hipGetLastError();
    }
    switch (M) {
    case 128: fused_vol_inv<8>(casVol, V, pad, vol, N, precomp, a, b, zeroNyquist, sc, s); break;
    case 192: fused_vol_inv<12>(casVol, V, pad, vol, N, precomp, a, b, zeroNyquist, sc, s); break;
    case 256: fused_vol_inv<16>(casVol, V, pad, vol, N, precomp, a, b, zeroNyquist, sc, s); break;
    case 384: fused_vol_inv<24>(casVol, V, pad, vol, N, precomp, a, b, zeroNyquist, sc, s); break;
    default: fused_vol_inv<32>(casVol, V, pad, vol, N, precomp, a, b, zeroNyquist, sc, s); break;
    }
    return hipGetLastError();
}

hipError_t launch_vol_to_real3d(const float *vol, int N, float *real, int M, const float *precomp,
                                hipStream_t s)
{
    const size_t total = (size_t)M * M * M;
    hipLaunchKernelGGL(k_vol_to_real3d, dim3(grid_for(total)), dim3(kThreads), 0, s, vol, N, real, M,
                       precomp, total);
    return hipGetLastError();
}

hipError_t launch_herm3d_to_casvol(const float2 *herm, int M, float *casVol, int V, int pad,
                                   hipStream_t s)
{
    const size_t total = (size_t)V * V * V;
    const float gsign = ((3 * (M / 2)) & 1) ? -1.f : 1.f;
    hipLaunchKernelGGL(k_herm3d_to_casvol, dim3(grid_for(total)), dim3(kThreads), 0, s, herm, M, casVol,
                       V, pad, gsign, total);
    return hipGetLastError();
}

hipError_t launch_casvol_to_herm3d(const float *casVol, int V, int pad, float2 *herm, int M,
                                   int zeroNyquist, hipStream_t s)
{
    const size_t total = (size_t)M * M * (M / 2 + 1);
    hipLaunchKernelGGL(k_casvol_to_herm3d, dim3(grid_for(total)), dim3(kThreads), 0, s, casVol, V, pad,
                       herm, M, zeroNyquist, total);
    return hipGetLastError();
}

hipError_t launch_real3d_to_vol(const float *real, int M, float *vol, int N, const float *precomp,
                                float scale, hipStream_t s)
{
    const size_t total = (size_t)N * N * N;
    const double gsign = ((3 * (M / 2)) & 1) ? -1.0 : 1.0;
    hipLaunchKernelGGL(k_real3d_to_vol, dim3(grid_for(total)), dim3(kThreads), 0, s, real, M, vol, N,
                       precomp, gsign * (double)scale, total);
    return hipGetLastError();
}

hipError_t launch_reduce_partials(float *out, const float *parts, int nParts, size_t n,
                                  size_t stride, int accumulate, hipStream_t s)
{
    if (!n) return hipSuccess;
    hipLaunchKernelGGL(k_reduce_partials, dim3(grid_for(n)), dim3(kThreads), 0, s, out, parts, nParts, n,
                       stride, accumulate);
    return hipGetLastError();
}

hipError_t launch_divide_density(float *out, const float *num, const float *den, size_t n,
                                 double eps, hipStream_t s)
{
    if (!n) return hipSuccess;
    hipLaunchKernelGGL(k_divide_density, dim3(grid_for(n)), dim3(kThreads), 0, s, out, num, den, n, eps);
    return hipGetLastError();
}

hipError_t launch_convert_volume(void *dst, int dtype, const float *src, size_t n, hipStream_t s)
{
    if (!n) return hipSuccess;
    if (dtype == DT_BF16)
        hipLaunchKernelGGL(k_to_bf16, dim3(grid_for(n)), dim3(kThreads), 0, s, (uint16_t *)dst, src, n);
    else if (dtype == DT_F16)
        hipLaunchKernelGGL(k_to_f16, dim3(grid_for(n)), dim3(kThreads), 0, s, (uint16_t *)dst, src, n);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t launch_check_volume(const void *vol, int dtype, size_t n, const float *ker, int K, unsigned *check,
                               hipStream_t s)
{
    hipLaunchKernelGGL(k_check_table, dim3(1), dim3(kThreads), 0, s, ker, K, check, 1u);
    if (n == 0) return hipGetLastError();
    const dim3 grid(std::min(grid_for(n), 4096u)), block(kThreads);
    switch (dtype) {
    case DT_F32: hipLaunchKernelGGL(k_check_volume<DT_F32>, grid, block, 0, s, vol, n, check); break;
    case DT_BF16: hipLaunchKernelGGL(k_check_volume<DT_BF16>, grid, block, 0, s, vol, n, check); break;
    case DT_F16: hipLaunchKernelGGL(k_check_volume<DT_F16>, grid, block, 0, s, vol, n, check); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_fill(float *p, float value, size_t n, hipStream_t s)
{
    if (!n) return hipSuccess;
    hipLaunchKernelGGL(k_fill, dim3(grid_for(n)), dim3(kThreads), 0, s, p, value, n);
    return hipGetLastError();
}

hipError_t launch_filter_cas_to_complex(const float *in, float2 *out, int size, int nSlices,
                                        hipStream_t s)
{
    const int volumeMode = nSlices <= 0;
    const int slices = volumeMode ? size : nSlices;
    const size_t total = (size_t)size * size * slices;
    if (!total) return hipSuccess;
    hipLaunchKernelGGL(k_f_cas_to_complex, dim3(grid_for(total)), dim3(kThreads), 0, s, in, out, size,
                       slices, volumeMode, total);
    return hipGetLastError();
}

hipError_t launch_filter_complex_to_cas(const float2 *in, float *out, int size, int nSlices,
                                        hipStream_t s)
{
    const size_t n = (size_t)size * size * nSlices;
    if (!n) return hipSuccess;
    hipLaunchKernelGGL(k_f_complex_to_cas, dim3(grid_for(n)), dim3(kThreads), 0, s, in, out, n);
    return hipGetLastError();
}

hipError_t launch_filter_complex_to_real(const float2 *in, float *out, int size, int nSlices,
                                         hipStream_t s)
{
    const size_t n = (size_t)size * size * nSlices;
    if (!n) return hipSuccess;
    hipLaunchKernelGGL(k_f_complex_to_real, dim3(grid_for(n)), dim3(kThreads), 0, s, in, out, n);
    return hipGetLastError();
}

hipError_t launch_filter_real_to_complex(const float *in, float2 *out, int size, int nSlices,
                                         hipStream_t s)
{
    const size_t n = (size_t)size * size * nSlices;
    if (!n) return hipSuccess;
    hipLaunchKernelGGL(k_f_real_to_complex, dim3(grid_for(n)), dim3(kThreads), 0, s, in, out, n);
    return hipGetLastError();
}

hipError_t launch_filter_fftshift2d(void *data, int elemBytes, int size, int nSlices, hipStream_t s)
{
    if (size % 2) return hipErrorInvalidValue;
    const size_t total = (size_t)size * (size / 2) * nSlices;
    if (!total) return hipSuccess;
    if (elemBytes == 4)
        hipLaunchKernelGGL(k_f_fftshift2d<float>, dim3(grid_for(total)), dim3(kThreads), 0, s,
                           (float *)data, size, total);
    else if (elemBytes == 8)
        hipLaunchKernelGGL(k_f_fftshift2d<float2>, dim3(grid_for(total)), dim3(kThreads), 0, s,
                           (float2 *)data, size, total);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t launch_filter_fftshift3d(void *data, int elemBytes, int size, hipStream_t s)
{
    if (size % 2) return hipErrorInvalidValue;
    const size_t total = (size_t)size * size * (size / 2);
    if (!total) return hipSuccess;
    if (elemBytes == 4)
        hipLaunchKernelGGL(k_f_fftshift3d<float>, dim3(grid_for(total)), dim3(kThreads), 0, s,
                           (float *)data, size, total);
    else if (elemBytes == 8)
        hipLaunchKernelGGL(k_f_fftshift3d<float2>, dim3(grid_for(total)), dim3(kThreads), 0, s,
                           (float2 *)data, size, total);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t launch_filter_pad(const float *in, float *out, int inSize, int outSize, int nSlices,
                             hipStream_t s)
{
    if (outSize < inSize) return hipErrorInvalidValue;
    const size_t total = (size_t)outSize * outSize * nSlices;
    if (!total) return hipSuccess;
    hipLaunchKernelGGL(k_f_pad, dim3(grid_for(total)), dim3(kThreads), 0, s, in, out, inSize, outSize,
                       total);
    return hipGetLastError();
}

hipError_t launch_filter_crop(const void *in, void *out, int elemBytes, int inSize, int outSize,
                              int nSlices, hipStream_t s)
{
    if (outSize > inSize) return hipErrorInvalidValue;
    const size_t total = (size_t)outSize * outSize * nSlices;
    if (!total) return hipSuccess;
    if (elemBytes == 4)
        hipLaunchKernelGGL(k_f_crop<float>, dim3(grid_for(total)), dim3(kThreads), 0, s,
                           (const float *)in, (float *)out, inSize, outSize, total);
    else if (elemBytes == 8)
        hipLaunchKernelGGL(k_f_crop<float2>, dim3(grid_for(total)), dim3(kThreads), 0, s,
                           (const float2 *)in, (float2 *)out, inSize, outSize, total);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t launch_filter_divide_scalar(float *data, float scalar, size_t n, hipStream_t s)
{
    if (scalar == 0.f) return hipErrorInvalidValue;
    if (!n) return hipSuccess;
    hipLaunchKernelGGL(k_f_divide_scalar, dim3(grid_for(n)), dim3(kThreads), 0, s, data, scalar, n);
    return hipGetLastError();
}

hipError_t launch_filter_divide_volume(float *a, const float *b, size_t n, hipStream_t s)
{
    if (!n) return hipSuccess;
    hipLaunchKernelGGL(k_f_divide_volume, dim3(grid_for(n)), dim3(kThreads), 0, s, a, b, n);
    return hipGetLastError();
}

hipError_t launch_filter_multiply_volume(float *a, const float *b, size_t n, hipStream_t s)
{
    if (!n) return hipSuccess;
    hipLaunchKernelGGL(k_f_multiply_volume, dim3(grid_for(n)), dim3(kThreads), 0, s, a, b, n);
    return hipGetLastError();
}

hipError_t launch_filter_multiply_complex_volume(float2 *a, const float *b, size_t n, hipStream_t s)
{
    if (!n) return hipSuccess;
    hipLaunchKernelGGL(k_f_multiply_complex_volume, dim3(grid_for(n)), dim3(kThreads), 0, s, a, b, n);
    return hipGetLastError();
}

hipError_t launch_filter_add_volume(float *a, const float *b, size_t n, hipStream_t s)
{
    if (!n) return hipSuccess;
    hipLaunchKernelGGL(k_f_add_volume, dim3(grid_for(n)), dim3(kThreads), 0, s, a, b, n);
    return hipGetLastError();
}

}  // namespace mgg
