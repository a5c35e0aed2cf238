// Backprojection stage on the device (and the fused Masking epilogue).
//
// Reference: backProjectLinear / backProjectNearest / backProjectTex
// (Backprojection.cu:238-336) with the LUT and constants of
// Backprojection::processor (:115-148); mask kernel (Masking.cu:157-169).
//
// Linear kernel design (gfx950):
//  * A workgroup owns a TILE x TILE pixel tile; each thread PPT pixels of one
//    column.  Angles are processed in chunks of A.
//  * For each angle of the chunk the tile's detector coordinates t span
//    [t(corner_min), t(corner_max)] -- t = fma(yp, sin, xp*cos) is monotone
//    in x and y under IEEE rounding, so the corners bound every pixel exactly.
//    Only that window (W entries) of the sinogram row is staged in LDS, as
//    pairs (s[k], s[k+1] - s[k]) with zeros outside [0, D): the inner loop
//    needs no bounds checks and one 8-byte LDS read per update.
//  * Per update: t (1 fma), floor + convert, fraction, address, one
//    ds_read_b64, one add and one fma; FP32 accumulation in angle order.
//  * With the mask fused, tiles and waves entirely outside the inscribed
//    circle skip the angle loop and write the masking value.
#include "device_common.h"

#include <algorithm>
#include <climits>
#include <type_traits>
#include <vector>
#include <cmath>

#include "../host/tables.h"

namespace risa {

struct BpParams {
    int N, P, D;
    int cI;              // (int)(D * 0.5): detector index of t = 0
    float scale, norm, center;
    int mask;
    float maskingValue;
    int W;               // staged window entries per angle
    int tilesX;
    float invW;
    float out_scale;     // multiplies sum * norm (1/in_scale for FP16 input)
    int AE;              // angles per staged chunk
    int zx, zy;          // log2 of the tile grid's width / height for the XCD-aware order, or -1
    int xg;              // 1: slice groups dealt to XCDs whole, 2: heaviest tiles first (bp_work), set per launch
    const int* order;    // bp_work's dispatch order tables (4 of tilesX * tilesY ranks) or null
};

// The tile of workgroup b.  Workgroups are dealt round-robin to the chip's 8
// XCDs, each with its own L2, so workgroup b runs on XCD b % 8.  On a
// power-of-two tile grid the tiles of one XCD are a contiguous range of the
// Z (Morton) order -- a compact block of the image -- which shrinks the union
// of their sinogram windows, i.e. that XCD's L2 footprint and the HBM
// re-reads; other grids keep the row-major order.
__device__ __forceinline__ int2 bp_tile_of_rank(int r, const BpParams& p)
{
    if (p.zx < 0) return make_int2(r % p.tilesX, r / p.tilesX);
    int x = 0, y = 0, bit = 0;
    for (int i = 0; i < p.zx || i < p.zy; i++) {
        if (i < p.zx) x |= ((r >> bit++) & 1) << i;
        if (i < p.zy) y |= ((r >> bit++) & 1) << i;
    }
    return make_int2(x, y);
}
__device__ __forceinline__ int2 bp_tile_xy(int b, const BpParams& p)
{
    if (p.zx < 0) return make_int2(b % p.tilesX, b / p.tilesX);
    const int per = 1 << (p.zx + p.zy - 3);   // tiles per XCD (grid >= 8 tiles)
    return bp_tile_of_rank((b & 7) * per + (b >> 3), p);
}

// Tile and slice group of workgroup (blockIdx.x, blockIdx.y) of a grid of
// T = gridDim.x tiles x G = gridDim.y slice groups.  With p.xg = 1 (T a multiple
// of 8, and G a multiple or a divisor of 8) whole slice groups go to XCDs:
// workgroup L = x + y T runs on XCD L % 8 as that XCD's (L / 8)-th; for
// G >= 8 each XCD takes G / 8 groups, all their tiles; for G < 8, 8 / G XCDs
// share a group, each a contiguous range of its tile order.  One XCD's L2
// then holds few sinograms and each is fetched from HBM about once, where
// splitting every slice's tiles over all 8 XCDs fetches it up to 8 times.
// With p.xg = 2 the tiles go heaviest first over all XCDs, and without p.xg in
// the tile order of bp_tile_xy, group blockIdx.y either way.  Within an
// XCD's range the tiles are dispatched heaviest first when p.order is set
// (table lm = log2 of the XCDs per group: each range of T / 2^lm ranks
// sorted by the tile's pixels inside the mask), so the workgroups that end
// a launch are the light edge tiles, not the full ones; L2 locality does not
// depend on the order inside a range.
__device__ __forceinline__ int bp_work(const BpParams& p, int2& txy)
{
    if (!p.xg) {
        txy = bp_tile_xy(blockIdx.x, p);
        return blockIdx.y;
    }
    if (p.xg == 2) {   // heaviest first over all XCDs, group by group
        txy = bp_tile_of_rank(p.order[blockIdx.x], p);
        return blockIdx.y;
    }
    const int T = gridDim.x, G = gridDim.y;
    const long L = blockIdx.x + (long)blockIdx.y * T;
    const int xcd = (int)(L & 7);
    const long k = L >> 3;
    if (G >= 8) {
        const int rank = (int)(k % T);
        txy = bp_tile_of_rank(p.order ? p.order[rank] : rank, p);
        return xcd + 8 * (int)(k / T);
    }
    const int m = 8 / G;   // XCDs per group
    const int lm = m == 2 ? 1 : (m == 4 ? 2 : (m == 8 ? 3 : 0));
    const int rank = (xcd / G) * (T / m) + (int)k;
    txy = bp_tile_of_rank(p.order ? p.order[lm * T + rank] : rank, p);
    return xcd % G;
}
// The host's switch for bp_work.
static inline int xcd_groups(long tiles, long groups)
{
    return tiles % 8 == 0 && groups > 0 && (groups % 8 == 0 || 8 % groups == 0) ? 1 : 0;
}

// Detector coordinate of a pixel; the same operation sequence everywhere
// (backprojector, its window bounds, the adjoint projector).
__device__ __forceinline__ float bp_t(float xp, float yp, float c, float s)
{
    return __builtin_fmaf(yp, s, __fmul_rn(xp, c));
}

// A rounded product that multiply-add contraction cannot fuse into a
// following sum (under -ffp-contract=fast even __fmul_rn / __fadd_rn fuse:
// in HIP they are plain operators).  Only the sign of a zero product can
// differ from x * y, which no caller here observes.
__device__ __forceinline__ float rounded_mul(float x, float y)
{
    return __builtin_fmaf(x, y, 0.0f);
}

// Masking.cu:162-166: outside when the float distance exceeds N*N*0.25 (double).
// Rounded products and sum: symmetric in x and y.
__device__ __forceinline__ bool bp_outside(int x, int y, int N, float center)
{
    const float dX = (float)x - center, dY = (float)y - center;
    const float dist = rounded_mul(dX, dX) + rounded_mul(dY, dY);
    return (double)dist > (double)N * N * 0.25;
}

// floor(t) as an int in one instruction (v_cvt_flr_i32_f32); the compiler
// only selects it under finite-math assumptions, which this file does not
// make globally.
__device__ __forceinline__ int floor_to_int(float t)
{
    int k;
    asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(k) : "v"(t));
    return k;
}

// Splits t into the sample index floor(t) and the fraction t - floor(t)
// (the adjoint projector's split).
__device__ __forceinline__ void bp_split(float t, int& k, float& f)
{
    k = floor_to_int(t);
    f = __builtin_amdgcn_fractf(t);
}

// min(max(k, 0), hi) in one instruction (the compiler emits two).
__device__ __forceinline__ int clamp_index(int k, int hi)
{
    int r;
    asm("v_med3_i32 %0, %1, 0, %2" : "=v"(r) : "v"(k), "s"(hi));
    return r;
}

// LDS byte addresses: the per-angle row address (table base included) is
// staged once per chunk, so an update's LDS address is one v_lshl_add_u32.
typedef float lds_f2 __attribute__((ext_vector_type(2)));
typedef unsigned lds_u4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ unsigned lds_address(const void* p)
{
    return (unsigned)(size_t)(const __attribute__((address_space(3))) char*)p;
}
template <class T>
__device__ __forceinline__ T lds_load(unsigned addr)
{
    return *(const __attribute__((address_space(3))) T*)(size_t)addr;
}

// Per-tile preparation of one angle.
//
// t relative to an integer origin T (the floor of the tile's smallest t):
//   t' = fma(yp, sin, fma(xp, cos, -T)),
// monotone in x and y under IEEE rounding, so the tile corners bound it and
// the window of sample indices k' = floor(t') is [kmin', kmin' + W).  The
// absolute detector index of k' is k' + T + cI.
struct AngleWin {
    float c, s, negT;
    int kmin;   // kmin'
    int kabs;   // absolute detector index of kmin'
};

__device__ __forceinline__ AngleWin angle_window(float c, float s, float xa, float xb, float ya, float yb, int cI)
{
    const float tmin = fminf(fminf(bp_t(xa, ya, c, s), bp_t(xb, ya, c, s)),
                             fminf(bp_t(xa, yb, c, s), bp_t(xb, yb, c, s)));
    const float T = floorf(tmin);
    const float ua = __builtin_fmaf(xa, c, -T), ub = __builtin_fmaf(xb, c, -T);
    const float tm = fminf(fminf(__builtin_fmaf(ya, s, ua), __builtin_fmaf(ya, s, ub)),
                           fminf(__builtin_fmaf(yb, s, ua), __builtin_fmaf(yb, s, ub)));
    AngleWin w;
    w.c = c;
    w.s = s;
    w.negT = -T;
    w.kmin = floor_to_int(tm);
    w.kabs = w.kmin + (int)T + cI;
    return w;
}

// LDS layout of one tile: two row buffers of AE angles x W entries first
// (constant offset, so row addresses fold into the ds_read immediate), then
// info[P] = (cos, sin, -T, byte offset of k' = 0 of the angle's row) and
// kinfo[P] = (kmin', kabs).
//
// Staged entry of sample k' (w = k' - kmin'):  (e0, d) with
//   d = s[k+1] - s[k],  e0 = s[k] - k' d,   k = k' + T + cI
// (zeros outside [0, D)), so that s[k] + (t' - k') d = e0 + t' d and the
// update needs no fraction: acc += e0; acc = fma(t', d, acc).
//
// One tile of SB slices (1, 2 or 4), shared by the per-slice kernels and the
// persistent uneven-batch kernel.  All threads of the workgroup call it
// together.  in_f16: the sinogram is FP16 (value * in_scale; SB = 1 only).
// With SB > 1 the workgroup reconstructs the same tile of the nv <= SB
// slices sp[b] -> ip[b] (b < nv; sp[0] = sino_v, ip[0] = I) of one geometry: a
// staged entry holds every slice's pair (e0, d), so one 8 * SB-byte LDS
// read and one coordinate, floor and address serve SB updates, and each
// slice's arithmetic is exactly the one-slice tile's.
typedef float lds_f4 __attribute__((ext_vector_type(4)));
// Staged row buffers of a tile of SB slices per workgroup.
__host__ __device__ constexpr int bp_row_buffers(int sb) { return sb == 4 ? 1 : 2; }
// Four-slice entries are two 16-byte halves in two planes kQuadPlane bytes
// apart (slices 0-1, slices 2-3), so a wave's reads of either half are
// 16-byte strided like the two-slice tiles' (a 32-byte entry would put
// adjacent lanes' 16-byte reads 32 bytes apart) and both halves share one
// address, the second read taking the plane offset as its immediate.
constexpr unsigned kQuadPlane = 16384;
// LDS of one group of threads, a multiple of 16 B.
__host__ __device__ constexpr size_t tile_lds(int AE, int W, int sb)
{
    const size_t rows = sb == 4 ? (size_t)2 * kQuadPlane : (size_t)2 * AE * W * 8 * sb;
    return (rows + (size_t)3 * AE * 24 + 15) / 16 * 16;
}
template <int SB>
struct LdsEnt {
    float v[2 * SB];
};
template <int SB>
__device__ __forceinline__ LdsEnt<SB> lds_entry(unsigned addr)
{
    LdsEnt<SB> e;
    if constexpr (SB == 1) {
        const lds_f2 q = lds_load<lds_f2>(addr);
        e.v[0] = q[0];
        e.v[1] = q[1];
    } else {
#pragma unroll
        for (int i = 0; i < SB / 2; i++) {
            const lds_f4 q = lds_load<lds_f4>(addr + kQuadPlane * i);
#pragma unroll
            for (int j = 0; j < 4; j++) e.v[4 * i + j] = q[j];
        }
    }
    return e;
}
//
// Q > 1: Q groups of TX TY / PPT threads, group g over the angles
// [P g / Q, P (g + 1) / Q) with rows and windows of its own (LDS region g), the
// groups' sums added in order at the end.
template <int TX, int TY, int PPT, int E, int U, int SB = 1, int Q = 1>
__device__ __forceinline__ void bp_tile(const void* __restrict__ sino_v, float* __restrict__ I,
                                        const float* __restrict__ cosT, const float* __restrict__ sinT,
                                        const BpParams& p, int x0, int y0, int in_f16, char* smem,
                                        const float* const* sp = nullptr, float* const* ip = nullptr, int nv = 1)
{
    static_assert(SB == 1 || SB == 2 || SB == 4, "one, two or four slices per tile");
    // staged row buffers: two (the next chunk is committed while the current
    // one is read), one for four-slice tiles (their entries would otherwise
    // leave few angles per chunk; the commit then waits for a barrier after
    // the chunk is read)
    constexpr int NB = bp_row_buffers(SB);
    constexpr int NT = TX * TY / PPT;
    constexpr int RS = TY / PPT;
    constexpr unsigned EB = SB == 4 ? 16u : 8u * SB;   // entry stride in a row (a plane for SB = 4)
    static_assert(Q == 1 || NT % 64 == 0, "a wave works on one group's angles");
    const int grp = Q == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / NT);
    const int tid = Q == 1 ? (int)threadIdx.x : (int)threadIdx.x - grp * NT;
    const int tx = tid % TX, ty = tid / TX;
    const int pa = Q == 1 ? 0 : (int)((long)p.P * grp / Q), pb = Q == 1 ? p.P : (int)((long)p.P * (grp + 1) / Q);
    const float* S = reinterpret_cast<const float*>(sino_v);
    const uint16_t* S16 = reinterpret_cast<const uint16_t*>(sino_v);
    const int W = p.W, AE = p.AE;
    char* rows = Q == 1 ? smem : smem + grp * tile_lds(AE, W, SB);
    const unsigned rbase = lds_address(rows);
    float4* info = reinterpret_cast<float4*>(rows + (SB == 4 ? (size_t)2 * kQuadPlane : (size_t)NB * AE * W * EB));
    int2* kinfo = reinterpret_cast<int2*>(info + 3 * AE);

    const int x = x0 + tx;
    const float xp = ((float)x - p.center) * p.scale;
    float yp[PPT];
    bool use[PPT];
    int any = 0;
#pragma unroll
    for (int r = 0; r < PPT; r++) {
        const int y = y0 + ty + r * RS;
        yp[r] = ((float)y - p.center) * p.scale;
        const bool valid = x < p.N && y < p.N;
        use[r] = valid && !(p.mask && bp_outside(x, y, p.N, p.center));
        any |= use[r] ? 1 : 0;
    }
    if (!__syncthreads_or(any)) {
        if (Q > 1 && grp > 0) return;
#pragma unroll
        for (int r = 0; r < PPT; r++) {
            const int y = y0 + ty + r * RS;
            if (x < p.N && y < p.N) {
#pragma unroll
                for (int b = 0; b < SB; b++)
                    if (b < nv) (SB == 1 ? I : ip[b])[(long)y * p.N + x] = p.maskingValue;
            }
        }
        return;
    }
    const bool wave_active = __any(any);
    float acc[PPT][SB];
#pragma unroll
    for (int r = 0; r < PPT; r++)
#pragma unroll
        for (int b = 0; b < SB; b++) acc[r][b] = 0.0f;

    const float xa = ((float)x0 - p.center) * p.scale, xb = ((float)(x0 + TX - 1) - p.center) * p.scale;
    const float ya = ((float)y0 - p.center) * p.scale, yb = ((float)(y0 + TY - 1) - p.center) * p.scale;
    // the same number of chunks for every group: they share the barriers
    const int nch = ((p.P + Q - 1) / Q + AE - 1) / AE;
    // the windows of chunk ch go to ring slot ch % 3: chunk ch is computed
    // while ch + 1 is fetched and ch + 2 is prepared, one barrier per chunk
    // One thread per angle (AE <= 64 <= NT); its (cos, sin) is loaded well
    // before the window is computed.
    static_assert(NT >= 64, "a thread per angle of a chunk");
    auto load_angle = [&](int ch) {
        const int a = pa + ch * AE + tid;
        return tid < AE && a < pb ? make_float2(cosT[a], sinT[a]) : make_float2(0.0f, 0.0f);
    };
    auto make_info = [&](int ch, float2 cs) {
        if (tid >= min(AE, pb - pa - ch * AE)) return;
        const AngleWin w = angle_window(cs.x, cs.y, xa, xb, ya, yb, p.cI);
        const int row = (ch % NB) * AE * W + tid * W;
        info[(ch % 3) * AE + tid] = make_float4(w.c, w.s, w.negT, __uint_as_float(rbase + (unsigned)(row - w.kmin) * EB));
        kinfo[(ch % 3) * AE + tid] = make_int2(w.kmin, w.kabs);
    };
    {
        const float2 cs0 = load_angle(0), cs1 = load_angle(1);
        make_info(0, cs0);
        make_info(1, cs1);
    }
    __syncthreads();

    float s0r[E][SB], s1r[E][SB];
    bool in0r[E], in1r[E];
    int kr[E];
    auto fetch = [&](int ch) {
        const int p0 = pa + ch * AE, nae = min(AE, pb - p0) * W;
        const int2* kin = kinfo + (ch % 3) * AE;
#pragma unroll
        for (int q = 0; q < E; q++) {
            const int e = tid + q * NT;
            // (entries e >= nae are neither loaded nor committed)
            if (e < nae) {
                const int a = (int)(((float)e + 0.5f) * p.invW);
                const int w = e - a * W;
                const int2 ki = kin[a];
                const int k = ki.y + w;
                kr[q] = ki.x + w;
                // unconditional loads at clamped indices (inside row p0 + a),
                // zeroed outside [0, D); 32-bit offsets from the uniform base
                const unsigned row = __umul24((unsigned)(p0 + a), (unsigned)p.D);   // P, D < 2^24
                const unsigned i0 = row + (unsigned)clamp_index(k, p.D - 1);
                const unsigned i1 = row + (unsigned)clamp_index(k + 1, p.D - 1);
                if (SB == 1 && in_f16) {
                    const char* b = reinterpret_cast<const char*>(S16);
                    s0r[q][0] = half_bits_to_float(*reinterpret_cast<const uint16_t*>(b + i0 * 2u));
                    s1r[q][0] = half_bits_to_float(*reinterpret_cast<const uint16_t*>(b + i1 * 2u));
                } else {
#pragma unroll
                    for (int b = 0; b < SB; b++) {
                        if (b < nv) {
                            const char* base = reinterpret_cast<const char*>(SB == 1 ? S : sp[b]);
                            s0r[q][b] = *reinterpret_cast<const float*>(base + i0 * 4u);
                            s1r[q][b] = *reinterpret_cast<const float*>(base + i1 * 4u);
                        } else {
                            s0r[q][b] = 0.0f;
                            s1r[q][b] = 0.0f;
                        }
                    }
                }
                // zeroed at commit, so the loads stay in flight meanwhile
                in0r[q] = (unsigned)k < (unsigned)p.D;
                in1r[q] = (unsigned)(k + 1) < (unsigned)p.D;
            }
        }
    };
    auto commit = [&](int ch) {
        const int nae = min(AE, pb - pa - ch * AE) * W;
        char* buf = rows + (size_t)(ch % NB) * AE * W * EB;
#pragma unroll
        for (int q = 0; q < E; q++) {
            const int e = tid + q * NT;
            if (e < nae) {
                float ent[2 * SB];
#pragma unroll
                for (int b = 0; b < SB; b++) {
                    const float s0 = in0r[q] ? s0r[q][b] : 0.0f, s1 = in1r[q] ? s1r[q][b] : 0.0f;
                    const float d = s1 - s0;
                    ent[2 * b] = s0 - (float)kr[q] * d;
                    ent[2 * b + 1] = d;
                }
                if constexpr (SB == 1) {
                    reinterpret_cast<float2*>(buf)[e] = make_float2(ent[0], ent[1]);
                } else {
#pragma unroll
                    for (int i = 0; i < SB / 2; i++)
                        reinterpret_cast<float4*>(buf + kQuadPlane * i)[e] =
                            make_float4(ent[4 * i], ent[4 * i + 1], ent[4 * i + 2], ent[4 * i + 3]);
                }
            }
        }
    };
    // one update of slice b from the entry q at coordinate t
    auto update = [&](float& a, const LdsEnt<SB>& q, int b, float t) {
        a += q.v[2 * b];
        a = __builtin_fmaf(t, q.v[2 * b + 1], a);
    };

    fetch(0);
    commit(0);
    __syncthreads();
    for (int ch = 0; ch < nch; ch++) {
        const int na = min(AE, pb - pa - ch * AE);
        const float4* inf = info + (ch % 3) * AE;
        const float2 cs = load_angle(ch + 2);
        if (ch + 1 < nch) fetch(ch + 1);
        if (wave_active) {
            // U angles per step: all U*PPT LDS reads are issued before the
            // first accumulate so their latency overlaps
            int a = 0;
            for (; a + U <= na; a += U) {
                float4 in[U];
                float t[U][PPT];
                LdsEnt<SB> v[U][PPT];
#pragma unroll
                for (int u = 0; u < U; u++) in[u] = inf[a + u];
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const float xc = __builtin_fmaf(xp, in[u].x, in[u].z);
                    const unsigned bb = __float_as_uint(in[u].w);
#pragma unroll
                    for (int r = 0; r < PPT; r++) {
                        t[u][r] = __builtin_fmaf(yp[r], in[u].y, xc);
                        v[u][r] = lds_entry<SB>(bb + (unsigned)floor_to_int(t[u][r]) * EB);
                    }
                }
#pragma unroll
                for (int u = 0; u < U; u++)
#pragma unroll
                    for (int r = 0; r < PPT; r++)
#pragma unroll
                        for (int b = 0; b < SB; b++) update(acc[r][b], v[u][r], b, t[u][r]);
            }
            for (; a < na; a++) {
                const float4 in = inf[a];
                const float xc = __builtin_fmaf(xp, in.x, in.z);
                const unsigned bb = __float_as_uint(in.w);
#pragma unroll
                for (int r = 0; r < PPT; r++) {
                    const float t = __builtin_fmaf(yp[r], in.y, xc);
                    const LdsEnt<SB> q = lds_entry<SB>(bb + (unsigned)floor_to_int(t) * EB);
#pragma unroll
                    for (int b = 0; b < SB; b++) update(acc[r][b], q, b, t);
                }
            }
        }
        if constexpr (NB == 1) __syncthreads();   // the single row buffer is read
        if (ch + 1 < nch) commit(ch + 1);
        make_info(ch + 2, cs);
        __syncthreads();
    }
    if constexpr (Q > 1) {
        // the rows are read: the groups' sums go through their space
        float* red = reinterpret_cast<float*>(smem);
#pragma unroll
        for (int r = 0; r < PPT; r++)
#pragma unroll
            for (int b = 0; b < SB; b++)
                if (grp > 0) red[(((grp - 1) * PPT + r) * SB + b) * NT + tid] = acc[r][b];
        __syncthreads();
        if (grp > 0) return;
#pragma unroll
        for (int g = 0; g < Q - 1; g++)
#pragma unroll
            for (int r = 0; r < PPT; r++)
#pragma unroll
                for (int b = 0; b < SB; b++) acc[r][b] += red[((g * PPT + r) * SB + b) * NT + tid];
    }
#pragma unroll
    for (int r = 0; r < PPT; r++) {
        const int y = y0 + ty + r * RS;
        if (x < p.N && y < p.N) {
#pragma unroll
            for (int b = 0; b < SB; b++)
                if (b < nv)
                    (SB == 1 ? I : ip[b])[(long)y * p.N + x] =
                        use[r] ? acc[r][b] * p.norm * p.out_scale : p.maskingValue;
        }
    }
}

// Workgroup (x, y): tile x of slices SB*y .. SB*y + SB - 1 (those below `slices`).
// The slices of one launch: slice k is sino[k] -> img[k] (a contiguous batch
// fills the pointers by stride).
constexpr int kBpSlices = 64;
struct BpSlices {
    const float* sino[kBpSlices];
    float* img[kBpSlices];
};

template <int TX, int TY, int PPT, int E, int U, int SB, int Q>
__device__ __forceinline__ void bp_slices(const BpSlices& L, const float* __restrict__ cosT,
                                          const float* __restrict__ sinT, int slices, const BpParams& p)
{
    extern __shared__ __attribute__((aligned(16))) char smem[];
    int2 txy;
    const int first = bp_work(p, txy) * SB;
    const int x0 = txy.x * TX, y0 = txy.y * TY;
    if constexpr (SB == 1) {
        bp_tile<TX, TY, PPT, E, U, 1, Q>(L.sino[first], L.img[first], cosT, sinT, p, x0, y0, 0, smem);
    } else {
        const int nv = min(SB, slices - first);
        const float* sp[SB];
        float* ip[SB];
#pragma unroll
        for (int b = 0; b < SB; b++) {
            sp[b] = L.sino[b < nv ? first + b : first];
            ip[b] = L.img[b < nv ? first + b : first];
        }
        bp_tile<TX, TY, PPT, E, U, SB, Q>(sp[0], ip[0], cosT, sinT, p, x0, y0, 0, smem, sp, ip, nv);
    }
}

template <int TX, int TY, int PPT, int E, int U, int SB>
__global__ void __launch_bounds__(TX* TY / PPT) bp_linear_kernel(BpSlices L, const float* __restrict__ cosT,
                                                                 const float* __restrict__ sinT, int slices,
                                                                 BpParams p)
{
    bp_slices<TX, TY, PPT, E, U, SB, 1>(L, cosT, sinT, slices, p);
}

// The angles shared by Q groups of threads.
template <int TX, int TY, int PPT, int E, int U, int SB, int Q>
__global__ void __launch_bounds__(TX* TY / PPT* Q) bp_linear_groups_kernel(BpSlices L, const float* __restrict__ cosT,
                                                                           const float* __restrict__ sinT, int slices,
                                                                           BpParams p)
{
    bp_slices<TX, TY, PPT, E, U, SB, Q>(L, cosT, sinT, slices, p);
}

// A job of the persistent uneven batch (device copy of risa_bp_job + derived
// constants).
struct BpJobDev {
    const void* sino;
    float* img;
    int lut_off;
    int in_f16;
    BpParams p;
};

// Persistent backprojection over many geometries: a grid sized to the chip
// pulls tiles (sorted by cost, largest first) from an atomic counter until
// the list is exhausted; every workgroup reaches the exit.
template <int TX, int TY, int PPT, int E, int U>
__global__ void __launch_bounds__(TX* TY / PPT) bp_persistent_kernel(const BpJobDev* __restrict__ jobs,
                                                                     const int2* __restrict__ tiles, int ntiles,
                                                                     const float* __restrict__ cosT,
                                                                     const float* __restrict__ sinT,
                                                                     int* __restrict__ counter)
{
    extern __shared__ __attribute__((aligned(16))) char smem[];
    __shared__ int next;
    for (;;) {
        if (threadIdx.x == 0) next = atomicAdd(counter, 1);
        __syncthreads();
        const int t = next;
        __syncthreads();
        if (t >= ntiles) break;
        const int2 w = tiles[t];
        const BpJobDev& j = jobs[w.x];
        const int x0 = (w.y % j.p.tilesX) * TX, y0 = (w.y / j.p.tilesX) * TY;
        bp_tile<TX, TY, PPT, E, U>(j.sino, j.img, cosT + j.lut_off, sinT + j.lut_off, j.p, x0, y0, j.in_f16, smem);
    }
}

__global__ void reset_counter_kernel(int* counter) { *counter = 0; }

// FP16-sinogram variant over groups of 4 slices of one geometry.
//
// Input layout "x4": for slice group g, angle a and detector k the four
// slices' values are adjacent, halves[((g*P + a)*D + k)*4 + b] (value *
// in_scale); slices past the last one of the last group are zero.  The DFT-GEMM
// filter writes this layout directly.  Each staged LDS entry holds, per slice,
// the pair (s[k], s[k+1] - s[k]); one update of the 4 slices is one 16-byte
// LDS read, one v_cvt_pk_f16_f32 for the weight pair (1, f) and four
// v_dot2_f32_f16 into FP32 accumulators.  Same tiling, windows and chunked
// double buffering as bp_tile.
typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef float f2_t __attribute__((ext_vector_type(2)));

// (1, f) as an FP16 pair in one v_cvt_pk_f16_f32 (round to nearest even).
__device__ __forceinline__ h2_t weight_pair(float f)
{
    const f2_t v = {1.0f, f};
    return __builtin_convertvector(v, h2_t);
}

constexpr int kF16Group = 4;

struct HRow {
    h2_t v[kF16Group];
};

// (s[k], s[k+1]) of 4 slices (two 8-byte loads, zero outside [0, D)) ->
// the staged pairs (s[k], s[k+1] - s[k]); the difference is one FP16 rounding.
__device__ __forceinline__ HRow stage_pairs(uint2 q0, uint2 q1)
{
    const h2_t s01 = __builtin_bit_cast(h2_t, q0.x), s23 = __builtin_bit_cast(h2_t, q0.y);
    const h2_t d01 = __builtin_bit_cast(h2_t, q1.x) - s01, d23 = __builtin_bit_cast(h2_t, q1.y) - s23;
    HRow r;
    r.v[0] = h2_t{s01.x, d01.x};
    r.v[1] = h2_t{s01.y, d01.y};
    r.v[2] = h2_t{s23.x, d23.x};
    r.v[3] = h2_t{s23.y, d23.y};
    return r;
}

template <int G>
struct HRowG {
    HRow h[G];
};

// LDS of one group of threads: G planes of two chunks of E * threads 16-byte
// entries, and the ring of angle windows; a multiple of 16 B.
__host__ __device__ constexpr size_t f16_lds(int G, int E, int threads, int AE)
{
    return ((size_t)G * 2 * E * threads * 16 + (size_t)3 * AE * 24 + 15) / 16 * 16;
}

// G groups of 4 slices per workgroup: the per-pixel t, index and weight are
// shared by 4G slices.  Q groups of threads share the angles as in bp_tile.
template <int TX, int TY, int PPT, int E, int U, int G, int Q>
__device__ __forceinline__ void bp_f16_tile(const uint2* __restrict__ sino, float* __restrict__ img,
                                            const float* __restrict__ cosT, const float* __restrict__ sinT, int slices,
                                            const BpParams& p)
{
    constexpr int NT = TX * TY / PPT;
    constexpr int RS = TY / PPT;
    constexpr int B = kF16Group * G;
    using Entry = HRowG<G>;
    // one LDS plane per group of 4 slices, each two chunks of at most E*NT
    // 16-byte entries (AE*W <= E*NT): a group's reads stay 16-byte strided
    // (no bank conflicts) and the plane offset is a ds_read immediate
    constexpr int PLANE = 2 * E * NT;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int W = p.W, AE = p.AE;
    static_assert(NT % 64 == 0, "a wave works on one group's angles");
    const int grp = Q == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / NT);
    const int pa = Q == 1 ? 0 : (int)((long)p.P * grp / Q), pb = Q == 1 ? p.P : (int)((long)p.P * (grp + 1) / Q);
    char* region = Q == 1 ? smem : smem + grp * f16_lds(G, E, NT, AE);
    HRow* rows = reinterpret_cast<HRow*>(region);
    const unsigned rbase = lds_address(rows);
    float4* info = reinterpret_cast<float4*>(region + (size_t)G * PLANE * sizeof(HRow));
    int2* kinfo = reinterpret_cast<int2*>(info + 3 * AE);

    const int tid = (int)threadIdx.x - grp * NT;
    const int tx = tid % TX, ty = tid / TX;
    int2 txy;
    const int g0 = bp_work(p, txy) * G;
    const int x0 = txy.x * TX, y0 = txy.y * TY;
    const int ngroups = (slices + kF16Group - 1) / kF16Group;
    const int ng = min(G, ngroups - g0);
    const int b0 = g0 * kF16Group;
    const int nb = min(B, slices - b0);
    const uint2* S = sino + (long)g0 * p.P * p.D;
    const long gstride = (long)p.P * p.D;

    const int x = x0 + tx;
    const float xp = ((float)x - p.center) * p.scale;
    float yp[PPT];
    bool use[PPT];
    int any = 0;
#pragma unroll
    for (int r = 0; r < PPT; r++) {
        const int y = y0 + ty + r * RS;
        yp[r] = ((float)y - p.center) * p.scale;
        const bool valid = x < p.N && y < p.N;
        use[r] = valid && !(p.mask && bp_outside(x, y, p.N, p.center));
        any |= use[r] ? 1 : 0;
    }
    if (!__syncthreads_or(any)) {
        if (Q > 1 && grp > 0) return;
        for (int b = 0; b < nb; b++)
#pragma unroll
            for (int r = 0; r < PPT; r++) {
                const int y = y0 + ty + r * RS;
                if (x < p.N && y < p.N) img[(long)(b0 + b) * p.N * p.N + (long)y * p.N + x] = p.maskingValue;
            }
        return;
    }
    const bool wave_active = __any(any);
    float acc[PPT][B];
#pragma unroll
    for (int r = 0; r < PPT; r++)
#pragma unroll
        for (int b = 0; b < B; b++) acc[r][b] = 0.0f;

    const float xa = ((float)x0 - p.center) * p.scale, xb = ((float)(x0 + TX - 1) - p.center) * p.scale;
    const float ya = ((float)y0 - p.center) * p.scale, yb = ((float)(y0 + TY - 1) - p.center) * p.scale;
    // the same number of chunks for every group: they share the barriers
    const int nch = ((p.P + Q - 1) / Q + AE - 1) / AE;
    // one thread per angle (AE <= 64 <= NT), loaded well before its window
    auto load_angle = [&](int ch) {
        const int a = pa + ch * AE + tid;
        return tid < AE && a < pb ? make_float2(cosT[a], sinT[a]) : make_float2(0.0f, 0.0f);
    };
    auto make_info = [&](int ch, float2 cs) {
        if (tid >= min(AE, pb - pa - ch * AE)) return;
        const AngleWin w = angle_window(cs.x, cs.y, xa, xb, ya, yb, p.cI);
        const int row = (ch & 1) * AE * W + tid * W;
        info[(ch % 3) * AE + tid] = make_float4(
            w.c, w.s, w.negT, __uint_as_float(rbase + (unsigned)((row - w.kmin) * (int)sizeof(HRow))));
        kinfo[(ch % 3) * AE + tid] = make_int2(w.kmin, w.kabs);
    };
    {
        const float2 cs0 = load_angle(0), cs1 = load_angle(1);
        make_info(0, cs0);
        make_info(1, cs1);
    }
    __syncthreads();

    uint2 q0r[E][G], q1r[E][G];
    bool in0r[E], in1r[E];
    auto fetch = [&](int ch) {
        const int p0 = pa + ch * AE, nae = min(AE, pb - p0) * W;
        const int2* kin = kinfo + (ch % 3) * AE;
#pragma unroll
        for (int q = 0; q < E; q++) {
            const int e = tid + q * NT;
            // (entries e >= nae are neither loaded nor committed; groups
            // gi >= ng are loaded as zeros)
#pragma unroll
            for (int gi = 0; gi < G; gi++) {
                q0r[q][gi] = make_uint2(0u, 0u);
                q1r[q][gi] = make_uint2(0u, 0u);
            }
            if (e < nae) {
                const int a = (int)(((float)e + 0.5f) * p.invW);
                const int k = kin[a].y + e - a * W;
                // unconditional loads at clamped indices (inside row p0 + a),
                // zeroed outside [0, D); 32-bit byte offsets from each group's base
                const unsigned row = __umul24((unsigned)(p0 + a), (unsigned)p.D);   // P, D < 2^24
                const unsigned o0 = (row + (unsigned)clamp_index(k, p.D - 1)) * 8u;
                const unsigned o1 = (row + (unsigned)clamp_index(k + 1, p.D - 1)) * 8u;
                // zeroed at commit, so the loads stay in flight meanwhile
                in0r[q] = (unsigned)k < (unsigned)p.D;
                in1r[q] = (unsigned)(k + 1) < (unsigned)p.D;
#pragma unroll
                for (int gi = 0; gi < G; gi++) {
                    if (gi >= ng) break;
                    const char* b = reinterpret_cast<const char*>(S + gi * gstride);
                    q0r[q][gi] = *reinterpret_cast<const uint2*>(b + o0);
                    q1r[q][gi] = *reinterpret_cast<const uint2*>(b + o1);
                }
            }
        }
    };
    auto commit = [&](int ch) {
        const int nae = min(AE, pb - pa - ch * AE) * W;
        HRow* buf = rows + (ch & 1) * AE * W;
#pragma unroll
        for (int q = 0; q < E; q++) {
            const int e = tid + q * NT;
            if (e < nae) {
#pragma unroll
                for (int gi = 0; gi < G; gi++) {
                    const uint2 z = make_uint2(0u, 0u);
                    buf[gi * PLANE + e] = stage_pairs(in0r[q] ? q0r[q][gi] : z, in1r[q] ? q1r[q][gi] : z);
                }
            }
        }
    };
    fetch(0);
    commit(0);
    __syncthreads();
    for (int ch = 0; ch < nch; ch++) {
        const int na = min(AE, pb - pa - ch * AE);
        const float4* inf = info + (ch % 3) * AE;
        const float2 cs = load_angle(ch + 2);
        if (ch + 1 < nch) fetch(ch + 1);
        if (wave_active) {
            int a = 0;
            for (; a + U <= na; a += U) {
                float4 in[U];
                Entry v[U][PPT];
                h2_t wgt[U][PPT];
#pragma unroll
                for (int u = 0; u < U; u++) in[u] = inf[a + u];
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const float xc = __builtin_fmaf(xp, in[u].x, in[u].z);
                    const unsigned row = __float_as_uint(in[u].w);
#pragma unroll
                    for (int r = 0; r < PPT; r++) {
                        int k;
                        float f;
                        bp_split(__builtin_fmaf(yp[r], in[u].y, xc), k, f);
                        wgt[u][r] = weight_pair(f);
                        // 16-byte entries: one ds_read_b128 per group, 8 lanes per LDS cycle
                        const unsigned at = row + (unsigned)k * (unsigned)sizeof(HRow);
#pragma unroll
                        for (int gi = 0; gi < G; gi++)
                            v[u][r].h[gi] = __builtin_bit_cast(
                                HRow, lds_load<lds_u4>(at + gi * PLANE * (unsigned)sizeof(HRow)));
                    }
                }
#pragma unroll
                for (int u = 0; u < U; u++)
#pragma unroll
                    for (int r = 0; r < PPT; r++)
#pragma unroll
                        for (int b = 0; b < B; b++)
                            acc[r][b] = __builtin_amdgcn_fdot2(wgt[u][r], v[u][r].h[b / 4].v[b % 4], acc[r][b],
                                                               false);
            }
            for (; a < na; a++) {
                const float4 in = inf[a];
                const float xc = __builtin_fmaf(xp, in.x, in.z);
                const unsigned row = __float_as_uint(in.w);
#pragma unroll
                for (int r = 0; r < PPT; r++) {
                    int k;
                    float f;
                    bp_split(__builtin_fmaf(yp[r], in.y, xc), k, f);
                    const h2_t wgt = weight_pair(f);
                    const unsigned at = row + (unsigned)k * (unsigned)sizeof(HRow);
                    Entry v;
#pragma unroll
                    for (int gi = 0; gi < G; gi++)
                        v.h[gi] = __builtin_bit_cast(HRow,
                                                     lds_load<lds_u4>(at + gi * PLANE * (unsigned)sizeof(HRow)));
#pragma unroll
                    for (int b = 0; b < B; b++)
                        acc[r][b] = __builtin_amdgcn_fdot2(wgt, v.h[b / 4].v[b % 4], acc[r][b], false);
                }
            }
        }
        if (ch + 1 < nch) commit(ch + 1);
        make_info(ch + 2, cs);
        __syncthreads();
    }
    if constexpr (Q > 1) {
        float* red = reinterpret_cast<float*>(smem);   // the rows are read
#pragma unroll
        for (int r = 0; r < PPT; r++)
#pragma unroll
            for (int b = 0; b < B; b++)
                if (grp > 0) red[(((grp - 1) * PPT + r) * B + b) * NT + tid] = acc[r][b];
        __syncthreads();
        if (grp > 0) return;
#pragma unroll
        for (int g = 0; g < Q - 1; g++)
#pragma unroll
            for (int r = 0; r < PPT; r++)
#pragma unroll
                for (int b = 0; b < B; b++) acc[r][b] += red[((g * PPT + r) * B + b) * NT + tid];
    }
    for (int b = 0; b < nb; b++)
#pragma unroll
        for (int r = 0; r < PPT; r++) {
            const int y = y0 + ty + r * RS;
            if (x < p.N && y < p.N)
                img[(long)(b0 + b) * p.N * p.N + (long)y * p.N + x] =
                    use[r] ? acc[r][b] * p.norm * p.out_scale : p.maskingValue;
        }
}

template <int TX, int TY, int PPT, int E, int U, int G>
__global__ void __launch_bounds__(TX* TY / PPT) bp_linear_f16_kernel(const uint2* __restrict__ sino,
                                                                     float* __restrict__ img,
                                                                     const float* __restrict__ cosT,
                                                                     const float* __restrict__ sinT, int slices,
                                                                     BpParams p)
{
    bp_f16_tile<TX, TY, PPT, E, U, G, 1>(sino, img, cosT, sinT, slices, p);
}

// The angles shared by Q groups of threads.
template <int TX, int TY, int PPT, int E, int U, int G, int Q>
__global__ void __launch_bounds__(TX* TY / PPT* Q) bp_linear_f16_groups_kernel(const uint2* __restrict__ sino,
                                                                               float* __restrict__ img,
                                                                               const float* __restrict__ cosT,
                                                                               const float* __restrict__ sinT,
                                                                               int slices, BpParams p)
{
    bp_f16_tile<TX, TY, PPT, E, U, G, Q>(sino, img, cosT, sinT, slices, p);
}

// ---------------------------------------------------------------------------
// FP32 backprojection of 32 slices on the matrix cores, with both operands
// split into FP16 hi + lo parts (22 bits each).
//
// For one angle a 4 x 4 pixel block reads at most 8 consecutive samples of a
// sinogram row (scale <= kSplitMaxScale), each pixel two of them with weights
// 1 - f and f.  As a matrix product that is a 16 x 8 weight matrix, two
// entries per row, times the 8 samples of every slice; four angles side by
// side fill the K = 32 of v_mfma_f32_16x16x32_f16:
//   A [16 pixels][4 angles x 8 samples]: lane m + 16 g holds the 8 weights of
//     pixel m at angle g,
//   B [4 angles x 8 samples][16 slices]: lane n + 16 g the samples of slice n.
// Three products per 16 slices, hi hi + lo hi + hi lo, accumulate in FP32;
// the dropped lo lo term is 2^-24 of a product.
//
// Precision: of the operands' and the sums' rounding only the latter shows, 750
// additions to ever larger sums at 1000 angles.  Each block of 64 angles is
// therefore summed for itself and the blocks' sums are added up (32 registers,
// 32 additions per 64 angles).  Relative RMSE against float64 of a
// backprojection of filtered phantoms, by tile 32 x 32 / 16 x 16, and
// bp_linear_kernel's beside it: 512^2 x 1000 angles 2.68e-6 / 2.68e-6 (2.78e-6 /
// 2.76e-6; most of it is the angles' own FP32 rounding), 256^2 x 500 1.22e-6 /
// 1.20e-6 (1.35e-6 / 1.31e-6), 431 detectors on 501^2 x 776 8.4e-7 (1.09e-6),
// 504 on 454^2 x 763 1.47e-6 (1.61e-6); below it in all 11 geometries of 246 to
// 552 pixels tried.  As one running sum it was above it, by 1 to 11 per cent.
//
// The pixels' coordinates and weights cost the vector unit about 24 instructions
// per 64 (pixel, angle) pairs whatever the number of slices, where
// bp_linear_kernel spends 2.8 per pair and slice.
//
// Weight placement: with kb the block's first sample (an even detector, so
// two samples share a dword) and q = floor(t) - kb in [0, 6], the eight
// weights are the dword (1 - f, f) moved to half q of 16 bytes.  The four
// v_perm selectors that do it come from an LDS table indexed by q; a second,
// all-zero table serves the angles that pad the last group of four.
//
// The samples come packed by split_pack_kernel: per angle rows of two
// adjacent detectors, row R (detectors 2R, 2R + 1) being 32 dwords of hi
// pairs, one per slice, then 32 of lo pairs, with a zero row at either end.
// A chunk's rows go from global memory straight to LDS (16 bytes per lane, no
// registers or vector instructions); two row buffers, one barrier per chunk.
// An angle's rows are followed by 64 spare bytes, so that the two angles whose
// lanes are read together use different banks; every byte of a buffer belongs
// to one angle, since different waves copy them.  A block's 4 rows may run past
// its angle's rows: their weights are zero and what they hold is finite (the
// next angle's rows, or the zeroed bytes between angles and at the end of the
// buffer).
//
// Bound: issue, LDS reads beside it, and too few waves to fill either.  In a
// launch of 32 slices of 512^2 x 1000 angles the vector unit issues in 46 % of a
// SIMD's clocks and the matrix cores are busy in 28 %, the LDS in 45 % of a CU's
// (5 KB of operands per 64 (pixel, angle) pairs, no bank conflicts), and a wave
// waits for 43 % of its time.  Four waves per SIMD: the two sets of sums take 64
// registers, and six or eight waves would spill them.  512^2 x 1000 angles, 32
// slices with their packing (20 us), 32 x 32 / 32 x 16 / 16 x 16 tiles: 510 / 505
// / 524 us (624 and 790 for the smaller two with six and eight waves),
// bp_linear_kernel 745; 384^2 x 700 323 / 269 / 271 and 356.  Up to 16 slices
// read half of the samples and take 397 / 443 / 481 us without the packing, 32
// take 516 / 552 / 568.
// ---------------------------------------------------------------------------
typedef float f4_t __attribute__((ext_vector_type(4)));
typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
constexpr int kSplitSlices = 32;          // slices per workgroup
constexpr int kSplitRow = 256;            // bytes of a packed row
constexpr double kSplitMaxScale = 1.17;   // 3 sqrt(2) scale + 0.02 <= 5: q stays <= 6 after the alignment
constexpr int kSplitInfo = 128;           // ring of angle records
constexpr int kSplitSlack = 6;            // zeroed rows after a buffer

// Packed rows of one angle, the two zero rows included.
__host__ __device__ constexpr int split_rows(int D) { return (D + 1) / 2 + 2; }
// Staged rows of one angle, a multiple of the 4 a wave copies at once: W + 1
// samples from up to three before the window.
__host__ __device__ constexpr int split_staged(int W) { return ((W + 5) / 2 + 3) / 4 * 4; }
// Bytes from one staged angle to the next.
__host__ __device__ constexpr int split_pitch(int W) { return split_staged(W) * kSplitRow + 64; }
__host__ __device__ constexpr int split_buffer(int AE, int W) { return AE * split_pitch(W) + kSplitSlack * kSplitRow; }
// Selector tables (2 x 8 x 16 B), two row buffers, the angle records (16 + 16 B).
__host__ __device__ constexpr int split_lds(int AE, int W) { return 256 + 2 * split_buffer(AE, W) + kSplitInfo * 32; }

// x from lane 0 of each row of 16 lanes
__device__ __forceinline__ float row_first(float x)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x150, 0xf, 0xf, true));
}
// x minus the low (high) FP16 half of h in one instruction
__device__ __forceinline__ float less_low(float x, unsigned h)
{
    float r;
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h), "v"(x));
    return r;
}
__device__ __forceinline__ float less_high(float x, unsigned h)
{
    float r;
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h), "v"(x));
    return r;
}
// (a, b) as FP16 hi and lo pairs
__device__ __forceinline__ void split_pair(float a, float b, unsigned& hi, unsigned& lo)
{
    hi = __builtin_bit_cast(unsigned, __builtin_convertvector((f2_t{a, b}), h2_t));
    lo = __builtin_bit_cast(unsigned, __builtin_convertvector((f2_t{less_low(a, hi), less_high(b, hi)}), h2_t));
}

// [slices][P][D] FP32 -> packed rows (value * scale); workgroup (x, y): detectors
// 64 x .. 64 x + 63 of angle y; slices past the last one are written as zero.
__global__ void __launch_bounds__(256) split_pack_kernel(const float* __restrict__ sino, int slices, int P, int D,
                                                         float scale, unsigned* __restrict__ packed)
{
    __shared__ unsigned tile[32][65];
    const int p = blockIdx.y, RP = split_rows(D), R0 = 32 * blockIdx.x;
    unsigned* out = packed + (long)p * RP * 64;
    const bool vec = D % 4 == 0 && reinterpret_cast<uintptr_t>(sino) % 16 == 0;
    for (int i = threadIdx.x; i < kSplitSlices * 16; i += 256) {
        const int s = i / 16, r = 2 * (i % 16), k = 2 * (R0 + r);
        float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if (s < slices) {
            const float* row = sino + ((long)s * P + p) * D;
            if (vec && k + 3 < D) {
                const float4 f = *reinterpret_cast<const float4*>(row + k);
                v[0] = f.x; v[1] = f.y; v[2] = f.z; v[3] = f.w;
            } else {
#pragma unroll
                for (int j = 0; j < 4; j++)
                    if (k + j < D) v[j] = row[k + j];
            }
        }
#pragma unroll
        for (int j = 0; j < 2; j++)
            split_pair(v[2 * j] * scale, v[2 * j + 1] * scale, tile[r + j][s], tile[r + j][32 + s]);
    }
    __syncthreads();
    // row R of the sinogram is packed row R + 1
    for (int i = threadIdx.x; i < 32 * 16; i += 256) {
        const int r = i / 16, c = 4 * (i % 16);
        if (R0 + r < RP - 2)
            reinterpret_cast<uint4*>(out)[(R0 + r + 1) * 16 + i % 16] =
                make_uint4(tile[r][c], tile[r][c + 1], tile[r][c + 2], tile[r][c + 3]);
    }
    if (blockIdx.x == 0 && threadIdx.x < 32)
        reinterpret_cast<uint4*>(out)[(threadIdx.x < 16 ? 0 : (RP - 1) * 16) + threadIdx.x % 16] =
            make_uint4(0u, 0u, 0u, 0u);
}

// Test values for timing: zero mean, about a filtered sinogram's size.
__global__ void tune_fill_kernel(float* out, long n)
{
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        out[i] = (float)((int)((unsigned)i * 2654435761u) >> 8) * 0x1p-26f;
}

// The same in FP16, below 1/2 in magnitude.
__global__ void tune_fill_f16_kernel(uint16_t* out, long n)
{
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        out[i] = float_to_half_bits((float)((int)((unsigned)i * 2654435761u) >> 8) * 0x1p-24f);
}

// Workgroup x: a TX x TY tile of up to 16 NU slices (a slice's bits do not depend
// on NU); each wave an 8 x 8 pixel block as 2 x 2 blocks of 4 x 4.
using lds_bytes = __attribute__((address_space(3))) char;

template <int TX, int TY, int NU>
__global__ void __launch_bounds__(TX* TY, 4) bp_split_kernel(const unsigned* __restrict__ packed,
                                                             float* __restrict__ img, const float* __restrict__ cosT,
                                                             const float* __restrict__ sinT, int slices, BpParams p)
{
    constexpr int NT = TX * TY, NW = NT / 64;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int AE = p.AE, RW = split_staged(p.W), pitch = split_pitch(p.W), bufsz = split_buffer(AE, p.W);
    const int RP = split_rows(p.D);
    uint4* tab = reinterpret_cast<uint4*>(smem);
    char* rows = smem + 256;
    float4* info = reinterpret_cast<float4*>(rows + 2 * bufsz);   // (cos, sin, -T, LDS address of sample k = 0)
    // (offset to a block's smallest t, selector table, packed row of the first staged row, -)
    float4* info2 = info + kSplitInfo;

    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
    int2 txy;
    bp_work(p, txy);
    const int x0 = txy.x * TX, y0 = txy.y * TY;
    const int bx = x0 + (wave % (TX / 8)) * 8, by = y0 + (wave / (TX / 8)) * 8;   // the wave's block
    const int m = lane & 15, g = lane >> 4;
    float xp[2], yp[2];
    bool use = false;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        xp[i] = ((float)(bx + 4 * i + (m & 3)) - p.center) * p.scale;
        yp[i] = ((float)(by + 4 * i + (m >> 2)) - p.center) * p.scale;
    }
#pragma unroll
    for (int sb = 0; sb < 4; sb++) {
        const int x = bx + 4 * (sb & 1) + (m & 3), y = by + 4 * (sb >> 1) + (m >> 2);
        use |= x < p.N && y < p.N && !(p.mask && bp_outside(x, y, p.N, p.center));
    }
    const bool active = __any(use);
    const int nch = __syncthreads_or(use) ? (p.P + AE - 1) / AE : 0;

    f4_t acc[4][NU], sum[4][NU];   // of the current block of 64 angles, and of those before
#pragma unroll
    for (int sb = 0; sb < 4; sb++)
#pragma unroll
        for (int u = 0; u < NU; u++) acc[sb][u] = sum[sb][u] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
    auto add_block = [&]() {
#pragma unroll
        for (int sb = 0; sb < 4; sb++)
#pragma unroll
            for (int u = 0; u < NU; u++) {
                sum[sb][u] += acc[sb][u];
                acc[sb][u] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
            }
    };

    const unsigned rbase = lds_address(rows), tbase = lds_address(tab);
    // records of angles 64 b .. 64 b + 63 (AE divides 64), slot angle % 128, by
    // one wave, another one each time; those past the last angle repeat it
    // with the all-zero selector table
    auto make_info = [&](int b) {
        if (wave != b % NW) return;
        const int pa = 64 * b + lane, pc = min(pa, p.P - 1), r = pa % kSplitInfo;
        const int ch = pc / AE, a = pc - ch * AE;
        const float xa = ((float)x0 - p.center) * p.scale, xb = ((float)(x0 + TX - 1) - p.center) * p.scale;
        const float ya = ((float)y0 - p.center) * p.scale, yb = ((float)(y0 + TY - 1) - p.center) * p.scale;
        const AngleWin w = angle_window(cosT[pc], sinT[pc], xa, xb, ya, yb, p.cI);
        // the origin is moved down to an even detector
        const int odd = ((int)-w.negT + p.cI) & 1, first = (w.kmin + odd - 2) & ~1;
        info[r] = make_float4(w.c, w.s, w.negT + (float)odd,
                              __uint_as_float(rbase + (unsigned)((ch & 1) * bufsz + a * pitch - first * (kSplitRow / 2))));
        info2[r] = make_float4(3.0f * p.scale * (fminf(w.c, 0.0f) + fminf(w.s, 0.0f)) - 0.01f,
                               __uint_as_float(tbase + (pa < p.P ? 0u : 128u)),
                               __int_as_float((first + (int)-w.negT - odd + p.cI) / 2 + 1), 0.0f);
    };
    // chunk ch's rows into its buffer: a wave copies 4 rows (1 KB) at a time
    const int units = AE * RW / 4;
    auto stage = [&](int ch, lds_bytes* buf) {
        const int p0 = ch * AE, na = min(AE, p.P - p0);
        for (int i = wave; i < units; i += NW) {
            const int a = i / (RW / 4), r = 4 * (i - a * (RW / 4));
            if (a >= na) break;
            const int R = __float_as_int(info2[(p0 + a) % kSplitInfo].z) + r + lane / 16;
            const unsigned* src = packed + ((long)(p0 + a) * RP + clamp_index(R, RP - 1)) * 64 + (lane & 15) * 4;
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                             buf + a * pitch + r * kSplitRow, 16, 0, 0);
        }
    };
    if (nch) {
        for (int i = tid; i < 2 * bufsz / 16; i += NT) reinterpret_cast<uint4*>(rows)[i] = make_uint4(0u, 0u, 0u, 0u);
        if (tid < 16) {
            // row q of the first table: byte selectors that move (w0, w1) to half q
            unsigned sel[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int d = tid - 2 * j;
                sel[j] = d == 0 ? 0x03020100u : (d == -1 ? 0x0c0c0302u : (d == 1 ? 0x01000c0cu : 0x0c0c0c0cu));
                if (tid > 6) sel[j] = 0x0c0c0c0cu;
            }
            tab[tid] = make_uint4(sel[0], sel[1], sel[2], sel[3]);
        }
        make_info(0);
        make_info(1);
        __syncthreads();
        stage(0, (lds_bytes*)rows);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    }
    // next: the buffer of chunk ch + 1.  Nothing else touches it before the
    // barrier; without __restrict__ the compiler makes the first LDS read of
    // the chunk wait for the copies into it (256 frames of 512^2 x 1000
    // angles: 4.40 ms, 4.28 with it).
    auto chunk = [&](int ch, lds_bytes* __restrict__ next) __attribute__((always_inline)) {
        const int p0 = ch * AE, na = min(AE, p.P - p0);
        if (ch + 1 < nch) stage(ch + 1, next);
        if (active) {
            const float4* inf = info + p0 % kSplitInfo + g;
            for (int a = 0; a < na; a += 4) {
                const float4 in = inf[a], in2 = inf[a + kSplitInfo];
                const unsigned rb = __float_as_uint(in.w) + (unsigned)m * 4u, tb = __float_as_uint(in2.y);
                const float xc[2] = {__builtin_fmaf(xp[0], in.x, in.z), __builtin_fmaf(xp[1], in.x, in.z)};
#pragma unroll
                for (int sb = 0; sb < 4; sb++) {
                    const float t = __builtin_fmaf(yp[sb >> 1], in.y, xc[sb & 1]);
                    const int kb = floor_to_int(row_first(t) + in2.x) & ~1;
                    int k;
                    float f;
                    bp_split(t, k, f);
                    const lds_u4 sel = lds_load<lds_u4>(tb + (unsigned)(k - kb) * 16u);
                    unsigned at = rb + (unsigned)kb * (kSplitRow / 2);
                    unsigned hi, lo;
                    split_pair(1.0f - f, f, hi, lo);
                    lds_u4 bh[NU], bl[NU];
#pragma unroll
                    for (int u = 0; u < NU; u++) {
                        // opaque bases: each two-address read then fills two
                        // adjacent registers of one operand
                        asm("" : "+v"(at));
#pragma unroll
                        for (int j = 0; j < 4; j++) bh[u][j] = lds_load<unsigned>(at + kSplitRow * j);
                        at += 128;
                        asm("" : "+v"(at));
#pragma unroll
                        for (int j = 0; j < 4; j++) bl[u][j] = lds_load<unsigned>(at + kSplitRow * j);
                        at -= 64;
                    }
                    lds_u4 ah, al;
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        ah[j] = __builtin_amdgcn_perm(0u, hi, sel[j]);
                        al[j] = __builtin_amdgcn_perm(0u, lo, sel[j]);
                    }
                    auto mma = [](f4_t& c, lds_u4 a, lds_u4 b) {
                        c = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8_t, a),
                                                                   __builtin_bit_cast(h8_t, b), c, 0, 0, 0);
                    };
#pragma unroll
                    for (int u = 0; u < NU; u++) mma(acc[sb][u], al, bh[u]);
#pragma unroll
                    for (int u = 0; u < NU; u++) mma(acc[sb][u], ah, bl[u]);
#pragma unroll
                    for (int u = 0; u < NU; u++) mma(acc[sb][u], ah, bh[u]);
                }
            }
        }
    };
    for (int ch = 0; ch < nch; ch++) {
        // chunks ch and ch + 1 lie in blocks of 64 angles ch AE / 64 and the
        // next: the ring's other half is free for the block after
        if (ch > 0 && ch * AE % 64 == 0) {
            if (ch * AE + 64 < p.P) make_info(ch * AE / 64 + 1);
            add_block();
        }
        chunk(ch, (lds_bytes*)rows + ((ch + 1) & 1) * bufsz);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wave's part of chunk ch + 1 is in LDS
        __syncthreads();
    }
    add_block();
    // lane (n = m, g): pixels 4 g .. 4 g + 3 of a block (its row g), slice 16 u + n
#pragma unroll
    for (int sb = 0; sb < 4; sb++) {
        const int x = bx + 4 * (sb & 1), y = by + 4 * (sb >> 1) + g;
        if (y >= p.N || x >= p.N) continue;
        bool in[4];
#pragma unroll
        for (int v = 0; v < 4; v++) in[v] = !(p.mask && bp_outside(x + v, y, p.N, p.center));
#pragma unroll
        for (int u = 0; u < NU; u++) {
            if (16 * u + m >= slices) continue;
            float* o = img + (long)(16 * u + m) * p.N * p.N + (long)y * p.N + x;
            f4_t r;
#pragma unroll
            for (int v = 0; v < 4; v++) r[v] = in[v] ? sum[sb][u][v] * p.norm * p.out_scale : p.maskingValue;
            if (x + 4 <= p.N && reinterpret_cast<uintptr_t>(o) % 16 == 0) {
                *reinterpret_cast<f4_t*>(o) = r;
            } else {
#pragma unroll
                for (int v = 0; v < 4; v++)
                    if (x + v < p.N) o[v] = r[v];
            }
        }
    }
}

// ---------------------------------------------------------------------------
// FP16-sinogram backprojection of 64 slices on the matrix cores, bit for bit
// bp_linear_f16_kernel's of the 16 x 16 tiles: the same FP16 operands (1, f)
// and (s0, s1 - s0), t from the same 16 x 16 tile origins, one product pair per
// pixel, slice and angle, added in angle order (an MFMA adds the products of a
// row into the FP32 sum as v_dot2_f32_f16 adds its two; the zeros add nothing).
//
// A block of 32 pixels (4 x 8 or 8 x 4) meets at most 8 floors of t at an
// angle when its long side runs along the angle's iso-lines (near 45 degrees,
// where it meets 9, a second product takes floors 8 to 15).  With K = 16 halves
// = 8 (s, d) pairs, v_mfma_f32_32x32x16_f16 is
//   A [32 pixels][8 pairs]: lane m + 32 h holds (1, f) of pixel m at pair
//     floor(t) - kb - 4 h of four, zeros elsewhere,
//   B [8 pairs][32 slices]: lane n + 32 h the pairs kb + 4 h .. + 3 of slice n.
//
// The block shape follows the angle's class (|cos| >= |sin|: 4 wide, 8 tall;
// else 8 wide, 4 tall).  A wave holds an 8 x 8 square as two blocks; row m =
// 16 e + 4 py + px of a block (px, py < 4, e the block's second 4 pixels along
// its long side) makes the change of shape a change of registers: the
// upper half of block 0's sums and the lower half of block 1's trade places.
//
// The pairs come packed by f16_pack_kernel, rows of one detector and 64
// slices; a chunk's rows go from global memory straight to LDS (two buffers,
// one barrier per chunk).  Rows are 288 bytes apart there, so that the rows
// the two halves of a wave read, four apart, use different banks.  A block may
// read rows past its angle's: their weights are zero and what they hold is
// finite unless a sample is not.  A non-finite sample meets the zero weights
// of its neighbours as NaN: a wave that ends with a non-finite sum evaluates
// its pixels again one by one (bp_f16_pixel).
//
// Bound: issue and LDS latency under load (vector issue in 47 % of a SIMD's
// clocks, matrix cores busy in 28 %, LDS in 42 % of a CU's without conflicts, a
// wave waiting for 46 % of its time).  A wave spends about 65
// instructions, 6.4 KB of LDS reads and 4 products per angle on 64 pixels of 64
// slices (bp_linear_f16_kernel 1.4 vector operations and 4 bytes of LDS per
// pixel and slice), so the 64 slices share what a pixel costs; the sums take
// half of the registers, which leaves four waves per SIMD, and the rows one
// workgroup per CU.  512^2 x 1000 angles, 64 slices: 705 us with the packing
// (45), 895 with bp_linear_f16_kernel.  Weights placed by compares instead of
// the selector table, and each wave copying rows of every angle: 784.
// ---------------------------------------------------------------------------
typedef float f16v_t __attribute__((ext_vector_type(16)));
constexpr int kPackSlices = 64;
constexpr int kPackInfo = 128;      // ring of angle records, per 16 x 16 part of the tile
constexpr int kPackPitch = 288;     // bytes between staged rows (18 16-byte pieces, the last two spare)
constexpr int kPackSlack = 5120;    // zeroed bytes after a buffer: 16 rows and more

// Packed rows of an angle: a zero row, detectors -1 .. D - 1, a zero row.
__host__ __device__ constexpr int pack_rows(int D) { return D + 3; }
// Staged rows of an angle: its window and two before (a block's first floor
// lies up to one below, and the parts' t round otherwise than the tile's).
__host__ __device__ constexpr int pack_staged(int W) { return W + 3; }
__host__ __device__ constexpr int pack_stride(int W) { return (pack_staged(W) * kPackPitch + 1023) / 1024 * 1024; }
__host__ __device__ constexpr int pack_buffer(int AE, int W) { return AE * pack_stride(W) + kPackSlack; }
__host__ __device__ constexpr int pack_lds(int AE, int W, int parts) { return 2 * pack_buffer(AE, W) + kPackInfo * 32 * parts + 28 * 16; }
// Products per block and angle.
__host__ __device__ inline int pack_steps(float c, float s, float scale)
{
    const float ac = fabsf(c), as = fabsf(s), span = scale * (3.0f * fmaxf(ac, as) + 7.0f * fminf(ac, as)) + 0.02f;
    return ((int)span + 2 + 7) / 8;   // floors a span can meet, eight per product
}

// x4 sinograms -> packed[P][pack_rows(D)][64] dwords (s, d), zero outside
// [0, D) and past the last group of 4 slices.  Bound by memory: 1000 x 512,
// 64 slices read 66 MB and write 132.
__global__ void __launch_bounds__(256) f16_pack_kernel(const uint2* __restrict__ sino, int groups, int P, int D,
                                                       uint4* __restrict__ packed)
{
    __shared__ uint2 tile[16][66];
    const int p = blockIdx.y, RP = pack_rows(D), R0 = 64 * blockIdx.x;
    for (int i = threadIdx.x; i < 16 * 65; i += 256) {
        const int g = i / 65, j = i - g * 65, k = R0 - 2 + j;
        tile[g][j] = g < groups && (unsigned)k < (unsigned)D ? sino[((long)g * P + p) * D + k] : make_uint2(0u, 0u);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 64 * 16; i += 256) {
        const int r = i / 16, g = i % 16;
        if (R0 + r < RP)
            packed[((long)p * RP + R0 + r) * 16 + g] =
                __builtin_bit_cast(uint4, stage_pairs(tile[g][r], tile[g][r + 1]));
    }
}

// Pixel (x, y) of one slice, sample by sample: row[4 k] is the slice's sample
// k of angle 0; xa .. yb the corners of its 16 x 16 tile.
__device__ __forceinline__ float bp_f16_pixel(const uint16_t* __restrict__ row, const float* __restrict__ cosT,
                                              const float* __restrict__ sinT, const BpParams& p, float xa, float xb,
                                              float ya, float yb, int x, int y)
{
    const float xq = ((float)x - p.center) * p.scale, yq = ((float)y - p.center) * p.scale;
    float acc = 0.0f;
#pragma unroll 1
    for (int a = 0; a < p.P; a++, row += (long)p.D * kF16Group) {
        const AngleWin w = angle_window(cosT[a], sinT[a], xa, xb, ya, yb, p.cI);
        int k;
        float f;
        bp_split(__builtin_fmaf(yq, w.s, __builtin_fmaf(xq, w.c, w.negT)), k, f);
        k += w.kabs - w.kmin;
        _Float16 h0 = (_Float16)0.0f, h1 = h0;
        if ((unsigned)k < (unsigned)p.D) h0 = __builtin_bit_cast(_Float16, row[(long)k * kF16Group]);
        if ((unsigned)(k + 1) < (unsigned)p.D) h1 = __builtin_bit_cast(_Float16, row[(long)(k + 1) * kF16Group]);
        acc = __builtin_amdgcn_fdot2(weight_pair(f), h2_t{h0, (_Float16)(h1 - h0)}, acc, false);
    }
    return acc;
}

// Workgroup x: a TX x TY tile of (up to) 64 slices, from `packed` (and the x4
// sinogram for non-finite pixels); each wave an 8 x 8 square.
template <int TX, int TY, int WPE>
__global__ void __launch_bounds__(TX* TY, WPE) bp_f16_mfma_kernel(const uint4* __restrict__ packed,
                                                                  const uint2* __restrict__ sino,
                                                                  float* __restrict__ img,
                                                                  const float* __restrict__ cosT,
                                                                  const float* __restrict__ sinT, int slices, BpParams p)
{
    constexpr int NT = TX * TY, NW = NT / 64, NB = 2, PX = TX / 16, PARTS = PX * (TY / 16), PITCH = kPackPitch;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int AE = p.AE, stride = pack_stride(p.W), bufsz = pack_buffer(AE, p.W), RP = pack_rows(p.D);
    char* rows = smem;
    float4* info = reinterpret_cast<float4*>(rows + 2 * bufsz);   // per part: (cos, sin, -T, LDS address of floor 0)
    // (offset to a block's smallest t, steps (negative: class B), packed row of staged row 0, -)
    int4* info2 = reinterpret_cast<int4*>(info + kPackInfo * PARTS);
    uint4* tab = reinterpret_cast<uint4*>(info2 + kPackInfo * PARTS);   // byte selectors that move (1, f) to pair q - 12

    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
    int2 txy;
    bp_work(p, txy);
    const int x0 = txy.x * TX, y0 = txy.y * TY;
    const int bx = x0 + (wave % (TX / 8)) * 8, by = y0 + (wave / (TX / 8)) * 8;   // the wave's square
    const int part = (bx - x0) / 16 + PX * ((by - y0) / 16);
    const int m = lane & 31, h = lane >> 5;
    bool use = false;
#pragma unroll
    for (int i = 0; i < 2; i++) {   // 32 of the square's pixels each
        const int x = bx + (m & 7), y = by + 4 * i + (m >> 3);
        use |= x < p.N && y < p.N && !(p.mask && bp_outside(x, y, p.N, p.center));
    }
    const bool active = __any(use);
    const int nch = __syncthreads_or(use) ? (p.P + AE - 1) / AE : 0;

    f16v_t acc[2][NB];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int u = 0; u < NB; u++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[i][u][v] = 0.0f;
    // the lane's pixel of the two blocks, for the current class
    float X[2], Y[2];
    int cls = 0;
    auto set_class = [&](int c) {
        const int px = m & 3, py = m >> 2 & 3, e = 4 * (m >> 4);
#pragma unroll
        for (int i = 0; i < 2; i++) {
            X[i] = ((float)(bx + px + (c ? e : 4 * i)) - p.center) * p.scale;
            Y[i] = ((float)(by + py + (c ? 4 * i : e)) - p.center) * p.scale;
        }
        if (c != cls)
#pragma unroll
            for (int u = 0; u < NB; u++)
#pragma unroll
                for (int v = 0; v < 8; v++) {
                    const float t = acc[0][u][8 + v];
                    acc[0][u][8 + v] = acc[1][u][v];
                    acc[1][u][v] = t;
                }
        cls = c;
    };
    set_class(0);

    auto coord = [&](int x) { return ((float)x - p.center) * p.scale; };
    const unsigned rbase = lds_address(rows), tbase = lds_address(tab + 12), m4 = (unsigned)m * 4u;
    // records of angles 64 b .. 64 b + 63 (AE divides 64), slot angle % 128, one
    // part per wave, other waves each time
    auto make_info = [&](int b) {
        const int q = (wave + NW - PARTS * b % NW) % NW;
        if (q >= PARTS) return;
        const int pa = 64 * b + lane, pc = min(pa, p.P - 1), r = pa % kPackInfo;
        const int ch = pc / AE, a = pc - ch * AE;
        const int xs = x0 + 16 * (q % PX), ys = y0 + 16 * (q / PX);
        const AngleWin t = angle_window(cosT[pc], sinT[pc], coord(x0), coord(x0 + TX - 1), coord(y0), coord(y0 + TY - 1), p.cI);
        const AngleWin w = angle_window(cosT[pc], sinT[pc], coord(xs), coord(xs + 15), coord(ys), coord(ys + 15), p.cI);
        const bool tall = fabsf(w.c) >= fabsf(w.s);
        const float lc = fminf(w.c, 0.0f) * p.scale, ls = fminf(w.s, 0.0f) * p.scale;
        const int steps = pack_steps(w.c, w.s, p.scale), row0 = w.kabs - w.kmin - t.kabs + 2;   // staged row of floor 0
        info[q * kPackInfo + r] = make_float4(
            w.c, w.s, w.negT, __uint_as_float(rbase + (unsigned)((ch & 1) * bufsz + a * stride + row0 * PITCH)));
        info2[q * kPackInfo + r] = make_int4(
            __float_as_int((tall ? 3.0f * lc + 7.0f * ls : 7.0f * lc + 3.0f * ls) - 0.01f), tall ? steps : -steps, t.kabs, 0);
    };
    // chunk ch's rows into its buffer (NW / AE waves per angle), 1 KB at a time
    const int per = stride / 1024, wpa = NW / AE, sa = wave / wpa, sj = wave - sa * wpa;
    auto stage = [&](int ch, lds_bytes* buf) {
        const int pa = ch * AE + sa;
        if (pa >= p.P) return;
        const int row0 = __builtin_amdgcn_readfirstlane(info2[pa % kPackInfo].z);
        const char* base = reinterpret_cast<const char*>(packed) + (long)pa * RP * 256;
        unsigned o = (unsigned)(64 * sj + lane);   // 16-byte piece; o / 18 the row (o < 2000)
        buf += sa * stride + sj * 1024;
        for (int j = sj; j < per; j += wpa) {
            const unsigned r = __umul24(o, 3641u) >> 16;
            const unsigned at = ((unsigned)clamp_index(row0 + (int)r, RP - 1) * 16u + min(o - __umul24(r, 18u), 15u)) * 16u;
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(base + at), buf, 16, 0, 0);
            o += 64u * (unsigned)wpa;
            buf += wpa * 1024;
        }
    };
    if (nch) {
        for (int i = tid; i < 2 * bufsz / 16; i += NT) reinterpret_cast<uint4*>(rows)[i] = make_uint4(0u, 0u, 0u, 0u);
        if (tid < 28) {
            unsigned sel[4];
#pragma unroll
            for (int j = 0; j < 4; j++) sel[j] = tid - 12 == j ? 0x03020100u : 0x0c0c0c0cu;
            tab[tid] = make_uint4(sel[0], sel[1], sel[2], sel[3]);
        }
        make_info(0);
        make_info(1);
        __syncthreads();
        stage(0, (lds_bytes*)rows);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    }
    // next: the buffer of chunk ch + 1, which nothing else touches before the
    // barrier (as in bp_split_kernel)
    auto chunk = [&](int ch, lds_bytes* __restrict__ next) __attribute__((always_inline)) {
        const int p0 = ch * AE, na = min(AE, p.P - p0);
        if (ch + 1 < nch) stage(ch + 1, next);
        if (!active) return;
        const float4* inf = info + part * kPackInfo + p0 % kPackInfo;
        const int4* inf2 = info2 + part * kPackInfo + p0 % kPackInfo;
        float4 in = inf[0];
        int2 in2 = *reinterpret_cast<const int2*>(inf2);
        for (int a = 0; a < na; a++) {
            const int st = __builtin_amdgcn_readfirstlane(in2.y);
            if ((st < 0) != (cls != 0)) set_class(st < 0);
            const int steps = st < 0 ? -st : st;
            const float off = __int_as_float(in2.x);
            unsigned at[2], w[2], tq[2];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const float t = __builtin_fmaf(Y[i], in.y, __builtin_fmaf(X[i], in.x, in.z));
                // lane 0 holds the block's first pixel
                const float t0 = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(t)));
                const int kb = floor_to_int(t0 + off) + 4 * h;
                int k;
                float f;
                bp_split(t, k, f);
                w[i] = __builtin_bit_cast(unsigned, weight_pair(f));
                tq[i] = tbase + (unsigned)(k - kb) * 16u;
                at[i] = __float_as_uint(in.w) + m4 + (unsigned)__mul24(kb, PITCH);
            }
            const int an = min(a + 1, na - 1);   // the next angle's record, while this one is multiplied
            in = inf[an];
            in2 = *reinterpret_cast<const int2*>(inf2 + an);
            for (int sp = 0;;) {
                lds_u4 B[2][NB], sel[2];
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    sel[i] = lds_load<lds_u4>(tq[i]);
#pragma unroll
                    for (int u = 0; u < NB; u++) {
                        asm("" : "+v"(at[i]));   // two-address reads of one operand
#pragma unroll
                        for (int j = 0; j < 4; j++) B[i][u][j] = lds_load<unsigned>(at[i] + PITCH * j);
                        at[i] += u + 1 < NB ? 128 : 8 * PITCH - 128 * (NB - 1);   // the next product's after the last
                    }
                }
                __builtin_amdgcn_sched_barrier(0);   // every read is under way before the first product
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    lds_u4 A;
#pragma unroll
                    for (int j = 0; j < 4; j++) A[j] = __builtin_amdgcn_perm(0u, w[i], sel[i][j]);
#pragma unroll
                    for (int u = 0; u < NB; u++)
                        acc[i][u] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                            __builtin_bit_cast(h8_t, A), __builtin_bit_cast(h8_t, B[i][u]), acc[i][u], 0, 0, 0);
                }
                if (__builtin_expect(++sp >= steps, 1)) break;
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    tq[i] -= 8 * 16;
                }
            }
        }
    };
    for (int ch = 0; ch < nch; ch++) {
        // chunks ch and ch + 1 lie in blocks of 64 angles ch AE / 64 and the
        // next: the ring's other half is free for the block after
        if (ch > 0 && ch * AE % 64 == 0 && ch * AE + 64 < p.P) make_info(ch * AE / 64 + 1);
        chunk(ch, (lds_bytes*)rows + ((ch + 1) & 1) * bufsz);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wave's part of chunk ch + 1 is in LDS
        __syncthreads();
    }
    set_class(0);
    // lane (n = m, h): register 8 e + 4 j + v of block i is pixel
    // (4 i + v, 4 e + 2 j + h) of the square, slice 32 u + n
    bool bad = false;
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int u = 0; u < NB; u++) {
            float z = 0.0f;
#pragma unroll
            for (int v = 0; v < 16; v++) z = __builtin_fmaf(acc[i][u][v], 0.0f, z);
            bad |= !(z == 0.0f);
            if (32 * u + m >= slices) continue;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int x = bx + 4 * i, y = by + 2 * r + h;
                if (x >= p.N || y >= p.N) continue;
                float* o = img + (long)(32 * u + m) * p.N * p.N + (long)y * p.N + x;
                f4_t w;
#pragma unroll
                for (int v = 0; v < 4; v++)
                    w[v] = p.mask && bp_outside(x + v, y, p.N, p.center) ? p.maskingValue
                                                                         : acc[i][u][4 * r + v] * p.norm * p.out_scale;
                if (x + 4 <= p.N && reinterpret_cast<uintptr_t>(o) % 16 == 0) {
                    *reinterpret_cast<f4_t*>(o) = w;
                } else {
#pragma unroll
                    for (int v = 0; v < 4; v++)
                        if (x + v < p.N) o[v] = w[v];
                }
            }
        }
    if (__any(bad)) {
        const int xs = x0 + 16 * (part % PX), ys = y0 + 16 * (part / PX);
#pragma unroll 1
        for (int i = 0; i < 32 * NB; i++) {   // (pixel of the lane's rows, u)
            const int x = bx + (i & 7), y = by + 2 * (i >> 3 & 3) + h, sl = 32 * (i >> 5) + m;
            if (sl >= slices || x >= p.N || y >= p.N || (p.mask && bp_outside(x, y, p.N, p.center))) continue;
            const uint16_t* row = reinterpret_cast<const uint16_t*>(sino + (long)(sl / kF16Group) * p.P * p.D) + sl % kF16Group;
            img[(long)sl * p.N * p.N + (long)y * p.N + x] =
                bp_f16_pixel(row, cosT, sinT, p, coord(xs), coord(xs + 15), coord(ys), coord(ys + 15), x, y) * p.norm *
                p.out_scale;
        }
    }
}

// [slices][P][D] FP16 -> the x4 layout (zero-filled past the last slice).
__global__ void f16_to_x4_kernel(const uint16_t* __restrict__ in, uint2* __restrict__ out, int slices, long plane)
{
    const long ngroups = (slices + kF16Group - 1) / kF16Group;
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < ngroups * plane;
         i += (long)gridDim.x * blockDim.x) {
        const long g = i / plane, e = i - g * plane;
        uint16_t h[kF16Group];
#pragma unroll
        for (int b = 0; b < kF16Group; b++) {
            const long s = g * kF16Group + b;
            h[b] = s < slices ? in[s * plane + e] : (uint16_t)0;
        }
        out[i] = make_uint2((uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16));
    }
}

// Nearest-neighbour variants (backProjectNearest :305-336, backProjectTex
// :273-302), one thread per pixel.
__global__ void bp_nearest_kernel(const float* __restrict__ sino, float* __restrict__ img,
                                  const float* __restrict__ cosT, const float* __restrict__ sinT, BpParams p,
                                  int tex)
{
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int y = blockIdx.y * blockDim.y + threadIdx.y;
    if (x >= p.N || y >= p.N) return;
    float sum = 0.0f;
    if (tex) {
        // backProjectTex: __fadd_rn(xp * cos, fma(yp, sin, cI)) with the sum and
        // the product rounded separately, as CUDA's intrinsics guarantee
        const float cI = (float)(p.D * 0.5);
        const float xp = ((float)x - p.center) * p.scale, yp = ((float)y - p.center) * p.scale;
        for (int a = 0; a < p.P; a++) {
            const float u = rounded_mul(xp, cosT[a]), v = __builtin_fmaf(yp, sinT[a], cI);
            const int t = (int)(u + v);
            if (t >= 0 && t < p.D) sum += sino[(long)a * p.D + t];
        }
        sum = sum * p.norm;
    } else {
        const float sc = (float)p.N / (float)p.D;
        const float xp = (float)(((double)x - (p.N - 1.0) * 0.5) / (double)sc);
        const float yp = (float)(((double)y - (p.N - 1.0) * 0.5) / (double)sc);
        for (int a = 0; a < p.P; a++) {
            const int t = (int)(roundf(__builtin_fmaf(yp, sinT[a], __fmul_rn(xp, cosT[a]))) + (float)p.cI);
            if (t >= 0 && t < p.D) sum += sino[(long)a * p.D + t];
        }
        sum = (float)((double)sum * M_PI / p.P * (double)sc);
    }
    if (p.mask && bp_outside(x, y, p.N, p.center)) sum = p.maskingValue;
    img[(long)y * p.N + x] = sum;
}

// out[x][y] = in[y][x] for an N x N image, 32 x 32 tiles through LDS.
__global__ void __launch_bounds__(256) transpose_kernel(const float* __restrict__ in, float* __restrict__ out, int N)
{
    __shared__ float tile[32][33];
    const int bx = blockIdx.x * 32, by = blockIdx.y * 32;
    for (int r = threadIdx.y; r < 32; r += 8) {
        const int y = by + r, x = bx + threadIdx.x;
        if (y < N && x < N) tile[r][threadIdx.x] = in[(long)y * N + x];
    }
    __syncthreads();
    for (int r = threadIdx.y; r < 32; r += 8) {
        const int x = bx + r, y = by + threadIdx.x;
        if (y < N && x < N) out[(long)x * N + y] = tile[threadIdx.x][r];
    }
}

// Ray-driven projector: the exact transpose of bp_linear_kernel.
//
// A workgroup serves one angle and kAdjK consecutive detectors, kAdjDPL per lane;
// its kAdjWaves waves split the image lines (wave w takes lines w,
// w + kAdjWaves, ...) and their partial sums are added in wave order, so the
// result does not depend on scheduling.  Each pixel's t is formed exactly as the forward kernel
// forms it for the tile (TX x TY) the pixel falls in -- relative to that
// tile's integer origin T, tabulated per angle in LDS -- so the weights are
// the forward's own and <BP s, x> = <s, BP^T x> holds to accumulation
// rounding: pixel (x, y) with k = floor(t) + T + cI adds (1 - f) img to
// entry k and f img to entry k + 1; pixels outside the mask add nothing.
// Detector k gathers the pixels with t in [k - cI - 1, k - cI + 1): on each
// line, a run of about 2 / (|cos| scale) pixels, found from the line's
// coordinate with 1/64 pixel of slack (the few ulps between that solve and
// the tile-relative t).  Lines run along x when |cos| >= |sin|, else along y,
// read as rows of the transposed image imgT so a wave's loads stay close
// together.  ltx, lty: log2 tile edges.
constexpr int kAdjDPL = 2;             // detectors per lane: k0 + lane + 64 j
constexpr int kAdjWaves = 8;           // waves per workgroup, splitting the image lines
constexpr int kAdjK = 64 * kAdjDPL;     // detectors per workgroup

// One lane's sum over its detector k, wave walking lines wave, wave + 4, ...
// Per line the wave first evaluates every pixel of the span its 64 detectors
// reach, one pixel per lane (coalesced loads, each pixel once): k = floor(t) +
// T + cI and its two contributions (1 - f) v, f v go to the wave's LDS buffer
// (cap entries).  Each lane then adds up the contributions to its detector
// along its own run of the span.  AX: lines run along x (rows of img); else
// along y (rows of imgT).  [SpLo, SpHi]: the span's bounds before the line's
// term, [Alo, Ahi]: the lane's run's.
template <bool AX>
__device__ __forceinline__ void adj_gather(const BpParams& p, const int2* inside, const float2* origin,
                                           const float* __restrict__ src, float c, float s, const int (&k)[kAdjDPL],
                                           float B, const float (&Alo)[kAdjDPL], const float (&Ahi)[kAdjDPL],
                                           float SpLo, float SpHi, int ltx, int lty, int wave, int lane, int* bk,
                                           float2* bv, int cap, float (&acc)[kAdjDPL])
{
#pragma unroll
    for (int j = 0; j < kAdjDPL; j++) acc[j] = 0.0f;
    for (int u = wave; u < p.N; u += kAdjWaves) {
        const float lc = ((float)u - p.center) * p.scale;
        const int2 in_u = inside[u];
        const int W0 = max(in_u.x, (int)floorf(__builtin_fmaf(-B, lc, SpLo)));
        const int W1 = min(min(in_u.y, (int)ceilf(__builtin_fmaf(-B, lc, SpHi))), W0 + cap - 1);
        if (W0 > W1) continue;   // the same for the whole wave
        const int trow = AX ? (u >> lty) * p.tilesX : (u >> ltx);
        const float* line = src + (long)u * p.N;
        for (int w = W0 + lane; w <= W1; w += 64) {
            const float2 o = origin[AX ? trow + (w >> ltx) : (w >> lty) * p.tilesX + trow];
            const float v = line[w];
            const float wp = ((float)w - p.center) * p.scale;
            const float tl = AX ? __builtin_fmaf(lc, s, __builtin_fmaf(wp, c, o.x))
                                : __builtin_fmaf(wp, s, __builtin_fmaf(lc, c, o.x));
            const float fl = floorf(tl);
            const float f = tl - fl;
            bk[w - W0] = (int)fl + __float_as_int(o.y);
            bv[w - W0] = make_float2((1.0f - f) * v, f * v);
        }
        // the buffer is the wave's own: LDS completes a wave's accesses in order
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int j = 0; j < kAdjDPL; j++) {
            const int r0 = max(W0, (int)floorf(__builtin_fmaf(-B, lc, Alo[j])));
            const int r1 = min(W1, (int)ceilf(__builtin_fmaf(-B, lc, Ahi[j])));
            for (int w = r0; w <= r1; w++) {
                const int kk = bk[w - W0];
                const float2 e = bv[w - W0];
                acc[j] += kk == k[j] ? e.x : (kk + 1 == k[j] ? e.y : 0.0f);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}

__global__ void __launch_bounds__(64 * kAdjWaves) bp_adjoint_kernel(const float* __restrict__ img,
                                                         const float* __restrict__ imgT, float* __restrict__ sino,
                                                         const float* __restrict__ cosT,
                                                         const float* __restrict__ sinT, BpParams p, int ltx, int lty,
                                                         int tilesY, int cap)
{
    extern __shared__ __attribute__((aligned(16))) char smem[];
    int2* inside = reinterpret_cast<int2*>(smem);                     // [N] per line: [lo, hi] inside the mask
    float2* origin = reinterpret_cast<float2*>(inside + p.N);         // per tile: (-T, bits of (int)T + cI)
    float* part = reinterpret_cast<float*>(origin + p.tilesX * tilesY);   // [waves][kAdjK]
    int* bk = reinterpret_cast<int*>(part + kAdjWaves * kAdjK);             // [waves][cap]
    float2* bv = reinterpret_cast<float2*>(bk + kAdjWaves * cap);           // [waves][cap]
    const int a = blockIdx.y, wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    const int k0 = blockIdx.x * kAdjK;
    int k[kAdjDPL];
#pragma unroll
    for (int j = 0; j < kAdjDPL; j++) k[j] = k0 + 64 * j + lane;
    const float c = cosT[a], s = sinT[a];
    const int TX = 1 << ltx, TY = 1 << lty;
    for (int t = threadIdx.x; t < p.tilesX * tilesY; t += blockDim.x) {
        const int x0 = (t % p.tilesX) * TX, y0 = (t / p.tilesX) * TY;
        const AngleWin aw = angle_window(c, s, ((float)x0 - p.center) * p.scale,
                                         ((float)(x0 + TX - 1) - p.center) * p.scale,
                                         ((float)y0 - p.center) * p.scale,
                                         ((float)(y0 + TY - 1) - p.center) * p.scale, p.cI);
        origin[t] = make_float2(aw.negT, __int_as_float((int)(-aw.negT) + p.cI));
    }
    for (int i = threadIdx.x; i < p.N; i += blockDim.x) {
        // the inside of line i is one interval around the centre (the test is
        // monotone in |x - center| and symmetric in x and y, so rows and
        // columns share it): found by bisection on the forward's own test
        int lo = 0, hi = p.N - 1;
        if (p.mask) {
            const int mid = (p.N - 1) / 2;
            if (bp_outside(mid, i, p.N, p.center)) {
                lo = 1;
                hi = 0;   // empty
            } else {
                int l = 0, r = mid;   // first inside column in [0, mid]
                while (l < r) {
                    const int m = (l + r) / 2;
                    if (bp_outside(m, i, p.N, p.center)) l = m + 1;
                    else r = m;
                }
                lo = l;
                l = mid;
                r = p.N - 1;   // last inside column in [mid, N - 1]
                while (l < r) {
                    const int m = (l + r + 1) / 2;
                    if (bp_outside(m, i, p.N, p.center)) r = m - 1;
                    else l = m;
                }
                hi = l;
            }
        }
        inside[i] = make_int2(lo, hi);
    }
    __syncthreads();
    const bool alongX = fabsf(c) >= fabsf(s);
    // on line u (coordinate up), t = w' cc + up ss with w' = (w - center) scale:
    // w = (t - up ss) / (cc scale) + center
    const float cc = alongX ? c : s, ss = alongX ? s : c;
    const float r = 1.0f / (cc * p.scale), B = ss * r;
    float Alo[kAdjDPL], Ahi[kAdjDPL];
#pragma unroll
    for (int j = 0; j < kAdjDPL; j++) {
        const float A0 = (float)(k[j] - p.cI - 1) * r + p.center, A1 = (float)(k[j] - p.cI + 1) * r + p.center;
        Alo[j] = fminf(A0, A1) - 0.015625f;
        Ahi[j] = fmaxf(A0, A1) + 0.015625f;
    }
    // the span of the workgroup's detectors k0 .. k0 + kAdjK - 1
    const float S0 = (float)(k0 - p.cI - 1) * r + p.center, S1 = (float)(k0 + kAdjK - p.cI) * r + p.center;
    const float SpLo = fminf(S0, S1) - 0.015625f, SpHi = fmaxf(S0, S1) + 0.015625f;
    int* wbk = bk + wave * cap;
    float2* wbv = bv + wave * cap;
    float acc[kAdjDPL];
    if (alongX)
        adj_gather<true>(p, inside, origin, img, c, s, k, B, Alo, Ahi, SpLo, SpHi, ltx, lty, wave, lane, wbk, wbv, cap,
                         acc);
    else
        adj_gather<false>(p, inside, origin, imgT, c, s, k, B, Alo, Ahi, SpLo, SpHi, ltx, lty, wave, lane, wbk, wbv,
                          cap, acc);
#pragma unroll
    for (int j = 0; j < kAdjDPL; j++) part[wave * kAdjK + 64 * j + lane] = acc[j];
    __syncthreads();
    for (int t = threadIdx.x; t < kAdjK; t += blockDim.x)
        if (k0 + t < p.D) {
            float sum = part[t];
            for (int w = 1; w < kAdjWaves; w++) sum += part[w * kAdjK + t];
            sino[(long)a * p.D + k0 + t] = sum * p.norm * p.out_scale;
        }
}

// ---------------------------------------------------------------------------
// Sheared-path adjoint projector: the exact transpose of bp_linear_kernel
// (the variant in use) without per-pixel scatter.
//
// For angle a write t(x, y) = (x - c0) cA + (r - c0) sA with c0 = (N-1)/2,
// where (cA, sA) = scale (cos, sin) and r = y when |cos| >= |sin| (class A,
// image read as is), else the roles of x and y swap (class B, the image read
// transposed) -- so |cA| >= |sA| and, for scale <= 1, |cA| <= 1.  Lane j of a
// wave follows the pixel path x = j + delta(r), delta(r) = -round(rho(r)),
// rho = (r - c0) sA / cA, one pixel per row r.  On that path the exact t is
// base_j + cA (rho - round rho), within |cA| / 2 <= 1/2 of base_j =
// (j - c0) cA, so its bin floor(t) takes at most two values, a_lo =
// floor(base_j - |cA|/2) and a_lo + 1, and the lane feeds at most the three
// bins a_lo .. a_lo + 2.
//
// The weights are the forward's own: per pixel the lane recomputes the
// forward's float coordinate t' = fma(yp, sin, fma(xp, cos, -T)) with T the
// integer origin of the pixel's forward tile (same operations, same tile
// table), so the forward's bin is a_lo + floor(u) with u = t' + T - a_lo
// (exact: an integer shift of a small float) and its fraction u - floor(u).
// With m = u - 1 in [-1, 1) a pixel of value v adds max(-m, 0) v to a_lo,
// (1 - |m|) v to a_lo + 1 and max(m, 0) v to a_lo + 2, so a lane keeps three
// sums over its path: sum v, sum v m and sum v |m| (|m| is a free source
// modifier of the FMA).  Only the pixel
// coordinate of the lane's axis and T vary along a path inside one forward
// tile row (class A) or column (class B); the wave tabulates them in LDS per
// such segment (class A: fma(xp, cos, -T) and T per pixel column; class B:
// yp and -T per pixel row), so a row costs one LDS read and 7 (class A) or
// 8 (class B) VALU operations per lane.  A pixel whose forward coordinate
// rounds across the lane's outer bin edges (|m| > 1 by ~1e-5) keeps weights
// off by that much: a set of measure ~1e-5 of the pixels.
//
// The paths of one angle tile every row exactly (bands of 64 lanes, J0 =
// -max|delta| + 64 b), so every pixel is on exactly one path per angle.
// Images are read from a zero-padded, masked copy (pixels outside the mask
// add nothing to the forward's output, so they are zero here) through buffer
// loads (hardware range check: an out-of-range offset reads 0).  A wave ends
// its path by adding its lanes' three contributions into a 72-entry LDS
// window of the bins its band covers and writing that window as a partial;
// adj_reduce_kernel sums a sinogram row's band partials in band order
// (deterministic).
// ---------------------------------------------------------------------------
constexpr int kAdjWin = 72;                 // bins per band window (64 |cA| + 3 <= 67)
constexpr int kAdjRec = kAdjWin + 1;        // record: kstart, then the window
constexpr int kAdjPad = 80;                 // zero columns either side of a padded image row
constexpr int kAdjWavesPerGroup = 8;        // angles per workgroup (one wave each), one band
constexpr int kAdjSlices = 16;              // images per pass through the buffers, in groups of 4 and a last 2 or 1
constexpr int kAdjPlaces = kAdjSlices + 3;  // padded copies: the groups of 4, one group of 2, one of 1
constexpr int kAdjTab = 192;                // segment table entries per wave (64 + 64 + 1 used at most)

struct AdjAngle {
    int p;          // angle index, -1: padding entry
    int cls;        // 0: read the image as is, 1: transposed
    float cA;       // along-lane coefficient (cos or sin), unscaled
    int J0base;     // -max|delta|
    int nb;         // bands of this angle
};

struct AdjParams {
    int N, P, D, cI;
    int PW;               // padded row length (N + 2 kAdjPad)
    int nbmax;            // bands per angle in the partial layout
    int npos;             // entries of the sorted angle list
    float scale, center;  // the forward's pixel coordinate ((float)x - center) * scale
    double c0;            // (N - 1) / 2
    float outmul;         // norm * out_scale
    long img_stride;      // elements per padded image
    int quads, tail;      // groups of four images of the pass, and the images of the group behind them (0 .. 2)
    int lgTX, lgTY;       // log2 of the forward tile's width / height
    int tilesX, tilesY;   // the forward's tile grid
};

// The forward's tile origins T[a][tile row][tile column] for tiles of
// TX x TY (bp_tile's angle_window on the same inputs) and its row
// coordinates ((float)r - center) * scale.
__global__ void adj_tile_origin_kernel(const float* __restrict__ cosT, const float* __restrict__ sinT, AdjParams q,
                                       float* __restrict__ T, float* __restrict__ coord)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < q.N) coord[i] = ((float)i - q.center) * q.scale;
    const long tiles = (long)q.tilesX * q.tilesY;
    if (i >= tiles * q.P) return;
    const int a = (int)(i / tiles);
    const int trow = (int)(i % tiles) / q.tilesX, tcol = (int)(i % tiles) % q.tilesX;
    const int x0 = tcol << q.lgTX, y0 = trow << q.lgTY;
    const float xa = ((float)x0 - q.center) * q.scale, xb = ((float)(x0 + (1 << q.lgTX) - 1) - q.center) * q.scale;
    const float ya = ((float)y0 - q.center) * q.scale, yb = ((float)(y0 + (1 << q.lgTY) - 1) - q.center) * q.scale;
    const AngleWin w = angle_window(cosT[a], sinT[a], xa, xb, ya, yb, q.cI);
    T[i] = -w.negT;
}

// A group of W images (4, or the pass's last 2 or 1) is stored pixel by pixel,
// the W values side by side, so that one load fetches a pixel of all of them.
// Groups of 4 start at kAdjSlices / 4 places of 4 image_strides; a group of 2
// and one of 1 have places of their own behind them, since the padding columns
// (zero from set-up) lie elsewhere for every W.
__host__ __device__ inline long adj_group_offset(int group, int W, long img_stride)
{
    return (W == 4 ? 4L * group : W == 2 ? (long)kAdjSlices : (long)kAdjSlices + 2) * img_stride;
}

// Zero-padded, masked copies of a pass's images [N][N], in groups: A [r]
// [kAdjPad + x] = img[r][x], B [r][kAdjPad + x] = img[x][r] (transposed), zero
// outside the mask.  The padding columns are zeroed once at set-up and never
// written.
__global__ void __launch_bounds__(256) adj_pad_kernel(const float* __restrict__ img, int slices,
                                                      float* __restrict__ A, float* __restrict__ B, int N, int PW,
                                                      int mask, float center, long img_stride, int quads, int tail)
{
    __shared__ float4 tile[32][33];
    const int z = blockIdx.z, W = z < quads ? 4 : tail, s0 = 4 * z;
    const float* I = img + (long)s0 * N * N;
    float* As = A + adj_group_offset(z, W, img_stride);
    float* Bs = B + adj_group_offset(z, W, img_stride);
    const int bx = blockIdx.x * 32, by = blockIdx.y * 32;
    auto put = [&](float* out, long at, float4 v) {
        if (W == 4) reinterpret_cast<float4*>(out)[at] = v;
        else if (W == 2) reinterpret_cast<float2*>(out)[at] = make_float2(v.x, v.y);
        else out[at] = v.x;
    };
    for (int r = threadIdx.y; r < 32; r += 8) {
        const int y = by + r, x = bx + threadIdx.x;
        float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if (y < N && x < N) {
            if (!(mask && bp_outside(x, y, N, center)))
#pragma unroll
                for (int k = 0; k < 4; k++)
                    if (s0 + k < slices) v[k] = I[(long)k * N * N + (long)y * N + x];
            put(As, (long)y * PW + kAdjPad + x, make_float4(v[0], v[1], v[2], v[3]));
        }
        tile[r][threadIdx.x] = make_float4(v[0], v[1], v[2], v[3]);
    }
    __syncthreads();
    for (int r = threadIdx.y; r < 32; r += 8) {
        const int x = bx + r, y = by + threadIdx.x;   // B row x, column y
        if (y < N && x < N) put(Bs, (long)x * PW + kAdjPad + y, tile[threadIdx.x][r]);
    }
}

__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One lane's path over rows [r0, r1] of angle p (class CLS) through the AS
// images of a group at once (rsrc); returns each image's three sums.  The
// path, its load, table entries, the pixel coordinate and the fraction are
// shared; each image adds three accumulations per row, with the same
// operations as a one-image path.  tab: this wave's segment table.  rt[r] =
// {4 x index of the path's row-r pixel of lane 0 in the padded image, minus
// J0 * 4; delta(r) * 8}.  Rows go in blocks of 8 (16 for one image), loads
// first; half of that where a segment has fewer rows left (a partial block's
// spare rows add zero).
template <int CLS, int AS>
__device__ __forceinline__ void adj_path(__amdgpu_buffer_rsrc_t rsrc, const int2* __restrict__ rt,
                                         const float* __restrict__ coord, const float* __restrict__ Tp,
                                         const AdjParams& q, float2* tab, int J0, int lane, int r0, int r1, float c,
                                         float s, float A1, float (&g0)[AS], float (&gm)[AS], float (&ga)[AS])
{
    // the segment: rows of one forward tile row (class A) or column (class B)
    const int sh = CLS ? q.lgTX : q.lgTY;
    const int voff = lane * 4 * AS, J04 = J0 * 4;
    const unsigned lane8 = lds_address(tab) + (unsigned)lane * 8u;
    unsigned lbase = lane8;   // lane8 - 8 * (the segment's smallest delta)
    // the row's table entry: one VALU add on a scalar byte offset (left to
    // itself the compiler re-associates the address into two)
    auto entry = [&](int d8) {
        unsigned a;
        asm("v_add_u32 %0, %1, %2" : "=v"(a) : "s"(d8), "v"(lbase));
        const lds_f2 w = lds_load<lds_f2>(a);
        return make_float2(w.x, w.y);
    };
    auto load = [&](float (&v)[AS], int off) {
        const int o = (int)((unsigned)(off + J04) * AS);
        if constexpr (AS == 4) {
            const f4_t w = __builtin_bit_cast(f4_t, __builtin_amdgcn_raw_buffer_load_b128(rsrc, voff, o, 0));
#pragma unroll
            for (int k = 0; k < 4; k++) v[k] = w[k];
        } else if constexpr (AS == 2) {
            const lds_f2 w = __builtin_bit_cast(lds_f2, __builtin_amdgcn_raw_buffer_load_b64(rsrc, voff, o, 0));
            v[0] = w.x;
            v[1] = w.y;
        } else {
            v[0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, voff, o, 0));
        }
    };
    auto row = [&](const float (&v)[AS], float2 e, float rc) {
        float tp, rm;
        if (CLS == 0) {
            tp = __builtin_fmaf(rc, s, e.x);                           // fma(yp, sin, xc)
            rm = e.y - A1;
        } else {
            tp = __builtin_fmaf(e.x, s, __builtin_fmaf(rc, c, e.y));   // fma(yp, sin, fma(xp, cos, -T))
            rm = -e.y - A1;
        }
        const float m = tp + rm;
#pragma unroll
        for (int k = 0; k < AS; k++) {
            g0[k] += v[k];
            gm[k] = __builtin_fmaf(v[k], m, gm[k]);
            ga[k] = __builtin_fmaf(v[k], fabsf(m), ga[k]);   // |m|: a source modifier, no extra operation
        }
    };
    // NB rows from r, of which the first `live` count (the rest re-read row
    // r + live - 1, in bounds, and add zero)
    auto block = [&](auto nb, int r, int live) {
        constexpr int NB = decltype(nb)::value;
        float v[NB][AS], rc[NB];
        float2 e[NB];
#pragma unroll
        for (int i = 0; i < NB; i++) {
            const int ri = r + min(i, live - 1);
            const int2 t = rt[ri];
            load(v[i], t.x);
#pragma unroll
            for (int k = 0; k < AS; k++)
                if (i >= live) v[i][k] = 0.0f;
            e[i] = entry(t.y);
            rc[i] = coord[ri];
        }
#pragma unroll
        for (int i = 0; i < NB; i++) row(v[i], e[i], rc[i]);
    };
    int r = r0;
    while (r <= r1) {
        const int segend = (((r >> sh) + 1) << sh) - 1;
        if (r == r0 || (r & ((1 << sh) - 1)) == 0) {
            const int re = min(r1, segend);
            const int da = rt[r].y >> 3, db = rt[re].y >> 3;   // delta is monotone in r
            const int dmin = min(da, db);
            const int n = 64 + abs(db - da);
            wave_lds_sync();
            for (int i = lane; i < n; i += 64) {
                const int pos = J0 + dmin + i;
                const float pc = ((float)pos - q.center) * q.scale;
                if (CLS == 0) {
                    const int tcol = min(max(pos >> q.lgTX, 0), q.tilesX - 1);
                    const float T = Tp[(r >> q.lgTY) * q.tilesX + tcol];
                    tab[i] = make_float2(__builtin_fmaf(pc, c, -T), T);
                } else {
                    const int trow = min(max(pos >> q.lgTY, 0), q.tilesY - 1);
                    const float T = Tp[trow * q.tilesX + (r >> q.lgTX)];
                    tab[i] = make_float2(pc, -T);
                }
            }
            lbase = lane8 - (unsigned)(dmin * 8);
            wave_lds_sync();
        }
        // rows left in this segment (segments are whole tile rows / columns)
        const int lim = min(r1, segend) - r + 1;
        constexpr int BIG = AS == 1 ? 16 : 8, SMALL = BIG / 2;
        if (lim >= BIG) {
            block(std::integral_constant<int, BIG>{}, r, BIG);
            r += BIG;
        } else {
            block(std::integral_constant<int, SMALL>{}, r, min(lim, SMALL));
            r += min(lim, SMALL);
        }
    }
}

// The path of angle p's band b through group z's W images, and the band's
// window of each of the first nv of them.
template <int W>
__device__ __forceinline__ void adj_band(const float* __restrict__ A, const float* __restrict__ B,
                                         float* __restrict__ partial, const int2* __restrict__ rowtab, int2 rr,
                                         const float* __restrict__ coord, const float* __restrict__ Ttab, float c,
                                         float s, const AdjAngle& an, const AdjParams& q, int b, int z, int nv,
                                         float2* tab, float* w, int lane)
{
    const int p = an.p, J0 = an.J0base + 64 * b;
    // this lane's bins a_lo .. a_lo + 2
    const double cAd = (double)an.cA * (double)q.scale;
    const double base = ((double)(J0 + lane) - q.c0) * cAd;
    const int a_lo = (int)floor(base - 0.5 * fabs(cAd));
    const float* img = (an.cls ? B : A) + adj_group_offset(z, W, q.img_stride);
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(img), (short)0, (int)(unsigned)(q.img_stride * 4 * W), 0x00020000);
    const int2* rt = rowtab + (long)p * q.N;
    const float* Tp = Ttab + (long)p * q.tilesX * q.tilesY;
    const float A1 = (float)(a_lo + 1);
    float g0[W], gm[W], ga[W];
#pragma unroll
    for (int k = 0; k < W; k++) g0[k] = gm[k] = ga[k] = 0.0f;
    if (an.cls) adj_path<1, W>(rsrc, rt, coord, Tp, q, tab, J0, lane, rr.x, rr.y, c, s, A1, g0, gm, ga);
    else adj_path<0, W>(rsrc, rt, coord, Tp, q, tab, J0, lane, rr.x, rr.y, c, s, A1, g0, gm, ga);
    // window of the band: the lanes' a_lo are monotone in the lane index
    const int kstart = min(__builtin_amdgcn_readfirstlane(a_lo), __builtin_amdgcn_readlane(a_lo, 63));
    const int wi = min(max(a_lo - kstart, 0), kAdjWin - 3);
#pragma unroll
    for (int k = 0; k < W; k++) {
        if (k >= nv) break;
        // the path's three contributions (t-bins a_lo, a_lo + 1, a_lo + 2):
        // max(-m, 0) = (|m| - m) / 2, 1 - |m|, max(m, 0) = (|m| + m) / 2
        const float c0v = 0.5f * (ga[k] - gm[k]), c1v = g0[k] - ga[k], c2v = 0.5f * (ga[k] + gm[k]);
        float* rec = partial + (((long)(4 * z + k) * q.P + p) * q.nbmax + b) * kAdjRec;
        for (int j = lane; j < kAdjWin; j += 64) w[j] = 0.0f;
        wave_lds_sync();
        atomicAdd(&w[wi], c0v);
        atomicAdd(&w[wi + 1], c1v);
        atomicAdd(&w[wi + 2], c2v);
        wave_lds_sync();
        if (lane == 0) rec[0] = __int_as_float(kstart);
        for (int j = lane; j < kAdjWin; j += 64) rec[1 + j] = w[j];
        wave_lds_sync();   // the window is read before the next image clears it
    }
}

// Workgroup (x, y, z): kAdjWavesPerGroup angles of the sorted list, band y,
// group z of the pass: four images for z < q.quads (QUADS), the last TAIL ones
// behind them.
//
// Bound by vector issue (one operation in 5.1 clocks per SIMD) and by the L1's
// accesses (in 86% of the clocks): a row of a wave costs 4 (class A) or 5
// operations, one load and one LDS read for the path and three operations per
// image.  Hence four images at once (16 operations for 256 image values; two
// at once 10 for 128), and the images stored side by side: one 16-byte load a
// lane instead of four.  16 images of 512^2 x 720 angles: 545 us, 741 with two
// images from separate planes; 5 images of 320^2 x 181 angles: 59 us, 76.
template <bool QUADS, int TAIL>
__global__ void __launch_bounds__(64 * kAdjWavesPerGroup) bp_adjoint_path_kernel(
    const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ partial,
    const AdjAngle* __restrict__ angles, const int2* __restrict__ bands, const int2* __restrict__ rowtab,
    const float* __restrict__ coord, const float* __restrict__ Ttab, const float* __restrict__ cosT,
    const float* __restrict__ sinT, int slices, AdjParams q)
{
    __shared__ float win[kAdjWavesPerGroup][kAdjWin];
    __shared__ float2 tabs[kAdjWavesPerGroup][kAdjTab];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int lane = threadIdx.x % 64;
    const int pos = blockIdx.x * kAdjWavesPerGroup + wave;
    if (pos >= q.npos) return;
    const AdjAngle an = angles[pos];
    if (an.p < 0 || (int)blockIdx.y >= an.nb) return;
    // bands centre-out: the long paths through the middle of the image are
    // dispatched first, the short edge bands fill in behind them
    const int i = blockIdx.y, mid = (an.nb - 1) / 2;
    const int b = (i & 1) ? mid + (i + 1) / 2 : mid - i / 2;
    const int2 rr = bands[an.p * q.nbmax + b];
    const float c = cosT[an.p], s = sinT[an.p];
    const int z = blockIdx.z;
    if (QUADS && z < q.quads)
        adj_band<4>(A, B, partial, rowtab, rr, coord, Ttab, c, s, an, q, b, z, min(4, slices - 4 * z), tabs[wave],
                    win[wave], lane);
    else if constexpr (TAIL != 0)
        adj_band<TAIL>(A, B, partial, rowtab, rr, coord, Ttab, c, s, an, q, b, z, TAIL, tabs[wave], win[wave], lane);
}

// sino[s][a][k] = outmul * sum over the angle's bands (in band order) of the
// band windows' entry for t-bin k - cI.  One workgroup per sinogram row: the
// row's band records are staged in LDS with coalesced loads first.
__global__ void __launch_bounds__(256) adj_reduce_kernel(const float* __restrict__ partial,
                                                         const int* __restrict__ nb_of, float* __restrict__ sino,
                                                         AdjParams q)
{
    extern __shared__ float recs[];
    const int p = blockIdx.x, sl = blockIdx.y;
    const int nb = nb_of[p];
    const float* src = partial + ((long)sl * q.P + p) * q.nbmax * kAdjRec;
    for (int i = threadIdx.x; i < nb * kAdjRec; i += 256) recs[i] = src[i];
    __syncthreads();
    for (int k = threadIdx.x; k < q.D; k += 256) {
        const int tb = k - q.cI;
        float sum = 0.0f;
        for (int b = 0; b < nb; b++) {
            const float* rb = recs + b * kAdjRec;
            const int i = tb - __float_as_int(rb[0]);
            if (i >= 0 && i < kAdjWin) sum += rb[1 + i];
        }
        sino[((long)sl * q.P + p) * q.D + k] = sum * q.outmul;
    }
}

// Standalone Masking (Masking.cu:113-144): optional min-max normalisation
// (two-pass reduction), then the circular mask.
__global__ void minmax_partial_kernel(const float* __restrict__ img, long n, float2* __restrict__ partial)
{
    __shared__ float smin[256], smax[256];
    float mn = INFINITY, mx = -INFINITY;
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        const float v = img[i];
        mn = fminf(mn, v);
        mx = fmaxf(mx, v);
    }
    smin[threadIdx.x] = mn;
    smax[threadIdx.x] = mx;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) {
            smin[threadIdx.x] = fminf(smin[threadIdx.x], smin[threadIdx.x + s]);
            smax[threadIdx.x] = fmaxf(smax[threadIdx.x], smax[threadIdx.x + s]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = make_float2(smin[0], smax[0]);
}

__global__ void mask_apply_kernel(float* __restrict__ img, int N, float center, float value, int normalize,
                                  const float2* __restrict__ partial, int nparts)
{
    float mn = 0.0f, diff = 1.0f;
    if (normalize) {
        float a = INFINITY, b = -INFINITY;
        for (int i = 0; i < nparts; i++) { a = fminf(a, partial[i].x); b = fmaxf(b, partial[i].y); }
        mn = a;
        diff = b - a;
    }
    const int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y * blockDim.y + threadIdx.y;
    if (x >= N || y >= N) return;
    float* v = img + (long)y * N + x;
    if (normalize) *v = (*v - mn) / diff;
    if (bp_outside(x, y, N, center)) *v = value;
}

}  // namespace risa

// ----------------------------------------------------------------------------
// Variants and handles
// ----------------------------------------------------------------------------
namespace risa {

// A variant: tile edge, pixels per thread, staged entries per thread (E)
// and the cap on angles per chunk.  The chunk holds AE = min(amax,
// E * threads / W) angles so one thread stages at most E entries.
struct BpVariant {
    int tx, ty, ppt, e, u, sb, amax;   // sb: slices per workgroup (1, 2 or 4)
    void (*fn)(BpSlices, const float*, const float*, int, BpParams);
    int q = 1;                         // groups of threads that share the angles
    int threads() const { return tx * ty / ppt; }   // of one group
    // a chunk holds at least one angle's window
    bool stages(int W) const { return W <= e * threads(); }
};

#define RISA_BPV(TX, TY, PPT, E, U, SB, AMAX) {TX, TY, PPT, E, U, SB, AMAX, bp_linear_kernel<TX, TY, PPT, E, U, SB>}
#define RISA_BPQ(TX, TY, PPT, E, U, SB, AMAX, Q) \
    {TX, TY, PPT, E, U, SB, AMAX, bp_linear_groups_kernel<TX, TY, PPT, E, U, SB, Q>, Q}
static const BpVariant kVariants[] = {
    RISA_BPV(32, 32, 4, 8, 4, 1, 64), RISA_BPV(32, 16, 2, 8, 4, 1, 64), RISA_BPV(16, 16, 1, 4, 4, 1, 64),
    RISA_BPV(32, 32, 8, 16, 2, 1, 64), RISA_BPV(64, 16, 4, 16, 4, 1, 64), RISA_BPV(32, 16, 4, 16, 4, 1, 64),
    RISA_BPV(16, 32, 2, 8, 4, 1, 64), RISA_BPV(32, 32, 4, 8, 2, 1, 64), RISA_BPV(16, 16, 2, 8, 4, 1, 64),
    RISA_BPV(32, 8, 1, 4, 4, 1, 64),
    // two slices per workgroup: one coordinate, floor, address and 16-byte LDS read per two updates;
    // half the staged entries per thread keep the doubled entries at ~33 KB of LDS per workgroup
    RISA_BPV(32, 32, 4, 4, 2, 2, 64), RISA_BPV(32, 32, 4, 4, 4, 2, 64), RISA_BPV(32, 16, 2, 4, 4, 2, 64),
    RISA_BPV(16, 16, 1, 2, 4, 2, 64),
    // four slices per workgroup: two planes of 16-byte half entries, one staged row buffer
    RISA_BPV(32, 32, 4, 4, 1, 4, 64), RISA_BPV(32, 32, 4, 4, 2, 4, 64), RISA_BPV(32, 16, 2, 4, 2, 4, 64),
    RISA_BPV(16, 16, 1, 2, 4, 4, 64),
    // The angles shared by q groups of threads: where one or a few slices leave
    // each SIMD with one wave or a few, whose chain of LDS reads then sets the
    // time (one wave takes about 100 clocks per angle, of which it issues for
    // 40).  More waves at the same tiles: 256^2 x 500 angles, one slice 32.5 ->
    // 14.3 us; 512^2 x 1000 one slice 80 -> 53, four 145 -> 133; 384^2 x 360
    // six slices 67 -> 60.  Full launches stay with the variants above
    // (512^2 x 720, 16 slices: 314 us, 321 at best with groups).
    RISA_BPQ(16, 16, 2, 4, 4, 1, 32, 4), RISA_BPQ(16, 16, 2, 4, 4, 1, 16, 8), RISA_BPQ(32, 32, 4, 4, 2, 1, 32, 4),
    RISA_BPQ(16, 16, 2, 4, 4, 2, 32, 4), RISA_BPQ(16, 16, 1, 2, 4, 2, 32, 2), RISA_BPQ(32, 32, 4, 4, 2, 2, 32, 2),
};
#undef RISA_BPV
#undef RISA_BPQ
static constexpr int kNumVariants = sizeof(kVariants) / sizeof(kVariants[0]);

struct BpF16Variant {
    int tx, ty, ppt, e, u, g, amax;
    void (*fn)(const uint2*, float*, const float*, const float*, int, BpParams);
    int q = 1;   // groups of threads that share the angles
};
#define RISA_BPH(TX, TY, PPT, E, U, G, AMAX) \
    {TX, TY, PPT, E, U, G, AMAX, bp_linear_f16_kernel<TX, TY, PPT, E, U, G>}
#define RISA_BPG(TX, TY, PPT, E, U, G, AMAX, Q) \
    {TX, TY, PPT, E, U, G, AMAX, bp_linear_f16_groups_kernel<TX, TY, PPT, E, U, G, Q>, Q}
// 16-pixel-wide tiles: the 16-byte LDS entries of a half-wave row then
// stay clear of bank conflicts; G groups of 4 slices share each pixel's
// weight.  The LDS planes take G * 2 * E * threads * 16 B, at most 32 KB
// here, leaving room for several workgroups per CU.
static const BpF16Variant kF16Variants[] = {
    RISA_BPH(16, 32, 2, 4, 2, 1, 64), RISA_BPH(16, 32, 2, 2, 2, 1, 64), RISA_BPH(16, 32, 4, 4, 2, 1, 64),
    RISA_BPH(16, 16, 1, 2, 4, 2, 64), RISA_BPH(16, 32, 2, 2, 2, 2, 64), RISA_BPH(16, 32, 4, 4, 2, 2, 64),
    RISA_BPH(16, 32, 4, 2, 2, 2, 64), RISA_BPH(16, 16, 1, 2, 2, 2, 64), RISA_BPH(16, 16, 1, 1, 2, 4, 64),
    RISA_BPH(16, 8, 1, 1, 2, 8, 64),
    // The angles shared by q groups of threads, for launches that leave a SIMD
    // few waves (as in the FP32 table): 512^2 x 1000 angles, 4 slices 148 ->
    // 102 us, 8 slices 178 -> 162; 256^2 x 500, 4 slices 59 -> 26, 16 slices
    // 67 -> 49.  From 16 slices of 512^2 the variants above are at least as fast.
    RISA_BPG(16, 32, 2, 2, 2, 1, 32, 4), RISA_BPG(16, 16, 1, 1, 4, 1, 32, 4), RISA_BPG(16, 16, 1, 2, 4, 2, 32, 2),
    RISA_BPG(16, 32, 2, 2, 2, 2, 32, 2), RISA_BPG(16, 16, 1, 1, 2, 2, 32, 4),
};
#undef RISA_BPH
#undef RISA_BPG
static constexpr int kNumF16Variants = sizeof(kF16Variants) / sizeof(kF16Variants[0]);

// Largest window a tx x ty tile needs for detector scale `scale`: the span of
// t over the tile is at most scale * ((tx-1)|c| + (ty-1)|s|)
// <= scale * sqrt((tx-1)^2 + (ty-1)^2), and floor(t_max) - floor(t_min) + 1
// <= ceil(span) + 2 (plus slack for rounding of t and of the table).
static int window_entries(int tx, int ty, float scale)
{
    const double diag = std::sqrt((double)(tx - 1) * (tx - 1) + (double)(ty - 1) * (ty - 1));
    return (int)std::ceil(diag * (double)scale * 1.00001 + 1e-2) + 2;
}

// Angles per chunk and the dynamic LDS bytes of a tile of sb slices per
// workgroup: 2 row buffers x AE x W entries of 8 * sb bytes (sb = 4: one
// buffer of two kQuadPlane-byte planes of 16-byte half entries) + a ring of
// 3 chunks of per-angle windows (16 B + 8 B per angle).
constexpr size_t kMaxLds = 64 * 1024;
// AE also shrinks so the tile fits the LDS budget (sb = 4: a plane).
static int chunk_angles(int threads, int e, int amax, int W, int sb = 1, int q = 1)
{
    int ae = std::min(amax, e * threads / W);
    if (sb == 4) ae = std::min<long>(ae, (long)kQuadPlane / (16L * W));
    else ae = std::min<long>(ae, (long)kMaxLds / q / (2L * W * 8 * sb + 88));
    return std::max(1, ae);
}

}  // namespace risa

struct risa_bp_s {
    int device = 0;
    risa_geom g{};
    risa::BpLut lut;
    risa::DeviceBuffer<float> cosT, sinT;
    int variant = 0;
    int variant_f16 = 0;
    bool fuse_mask = false;
    risa::DeviceBuffer<uint2> x4;   // staging for risa_hip_bp_run_f16's plain layout [kF16StageGroups][P][D]
    risa::DeviceBuffer<float> imgT;  // transposed image for the fallback adjoint [N][N]
    // sheared-path adjoint (scale <= 1): tables and per-pass buffers
    bool adj_path = false;
    bool adj_gather = false;                 // risa_hip_bp_adjoint_method(h, 1)
    risa::AdjParams adj{};
    int adj_groups = 0;                      // workgroups along the sorted angle list
    risa::DeviceBuffer<risa::AdjAngle> adj_angles;
    risa::DeviceBuffer<int2> adj_rows;       // [P][N] {(r * PW + pad + delta(r)) * 4, delta(r) * 8}
    risa::DeviceBuffer<int2> adj_bands;      // [P][nbmax] {first row, last row}
    risa::DeviceBuffer<int> adj_nb;          // [P]
    risa::DeviceBuffer<float> adj_imgA, adj_imgB;   // [kAdjPlaces][N][PW] padded, masked copies, in groups
    risa::DeviceBuffer<float> adj_partial;   // [kAdjSlices][P][nbmax][kAdjRec]
    risa::DeviceBuffer<float> adj_T;         // [P][tilesY][tilesX] the forward's tile origins (variant in use)
    risa::DeviceBuffer<float> adj_coord;     // [N] the forward's pixel coordinates
    // bp_work's heaviest-first dispatch tables per tile shape (FP32 variants,
    // then FP16 variants): offset into tile_order, or -1
    risa::DeviceBuffer<int> tile_order;
    std::vector<long> order_off;
};

namespace risa {
// risa_hip_bp_run_f16 converts and backprojects up to this many groups of 4
// slices per pass through the staging buffer allocated at create.
constexpr int kF16StageGroups = 4;
}  // namespace risa

using namespace risa;

// The kernels address a slice's sinogram with 32-bit byte offsets (up to
// 8 B per sample in the FP16 4-slice layout).
static void check_sino_size(int P, int D)
{
    if ((long)P * D * 8 >= (1L << 31))
        fail(RISA_ERR_UNSUPPORTED, "sinogram of %d x %d samples exceeds the kernels' 32-bit offsets", P, D);
}

// XCD-aware tile order on power-of-two grids of at least 8 tiles.
static void set_tile_order(BpParams& p, int tilesY)
{
    auto log2_exact = [](int v) {
        int l = 0;
        while ((1 << l) < v) l++;
        return (1 << l) == v ? l : -1;
    };
    p.zx = log2_exact(p.tilesX);
    p.zy = log2_exact(tilesY);
    if (p.zx < 0 || p.zy < 0 || p.zx + p.zy < 3) p.zx = p.zy = -1;
}

// bp_work's dispatch tables for a TX x TY tile grid (bp_tile_of_rank's rank
// order, host side): table lm holds, for each range of T / 2^lm consecutive
// ranks, the range's ranks sorted by the tile's pixels inside the image (and
// the mask), most first (ties in rank order).  Empty when T is not a
// multiple of 8 (bp_work then keeps the plain order).
static std::vector<int> dispatch_order(const BpParams& p, int TX, int TY, bool mask)
{
    const int tilesY = ceil_div(p.N, TY), T = p.tilesX * tilesY;
    std::vector<int> out;
    if (T % 8 != 0) return out;
    std::vector<long> cost((size_t)T);
    for (int r = 0; r < T; r++) {
        int tx = 0, ty = 0;
        if (p.zx < 0) {
            tx = r % p.tilesX;
            ty = r / p.tilesX;
        } else {
            int bit = 0;
            for (int i = 0; i < p.zx || i < p.zy; i++) {
                if (i < p.zx) tx |= ((r >> bit++) & 1) << i;
                if (i < p.zy) ty |= ((r >> bit++) & 1) << i;
            }
        }
        long c = 0;
        for (int y = ty * TY; y < std::min(p.N, ty * TY + TY); y++)
            for (int x = tx * TX; x < std::min(p.N, tx * TX + TX); x++) {
                const double dx = (double)((float)x - p.center), dy = (double)((float)y - p.center);
                if (!mask || dx * dx + dy * dy <= (double)p.N * p.N * 0.25) c++;
            }
        cost[(size_t)r] = c;
    }
    out.resize((size_t)4 * T);
    for (int lm = 0; lm < 4; lm++) {
        const int block = T >> lm;
        for (int b0 = 0; b0 < T; b0 += block) {
            int* o = out.data() + (size_t)lm * T + b0;
            for (int i = 0; i < block; i++) o[i] = b0 + i;
            std::stable_sort(o, o + block, [&](int a, int b) { return cost[(size_t)a] > cost[(size_t)b]; });
        }
    }
    return out;
}

static BpParams make_params(const risa_bp_s* h, int tx, int ty)
{
    check_sino_size(h->g.numberOfParallelProjections, h->g.numberOfParallelDetectors);
    BpParams p{};
    p.N = h->g.numberOfPixels;
    p.P = h->g.numberOfParallelProjections;
    p.D = h->g.numberOfParallelDetectors;
    p.cI = (int)(p.D * 0.5);
    p.scale = h->lut.scale;
    p.norm = h->lut.norm;
    p.center = h->lut.center;
    p.mask = h->fuse_mask ? 1 : 0;
    p.maskingValue = (float)h->g.maskingValue;
    p.W = window_entries(tx, ty, p.scale);
    p.tilesX = ceil_div(p.N, tx);
    set_tile_order(p, ceil_div(p.N, ty));
    p.invW = 1.0f / (float)p.W;
    p.out_scale = 1.0f;
    return p;
}

// Tables of the sheared-path adjoint (bp_adjoint_path_kernel) in double on
// the host: per angle its class, path shifts delta(r) and bands; per band the
// rows whose path segment meets the mask.  Applies when scale * max(|cos|,
// |sin|) <= 1 for every angle (a lane's t then stays within two bins);
// otherwise the handle keeps the gather adjoint.  The forward's tile origins
// depend on the variant in use and are rebuilt on the device per call.
static void setup_adjoint(risa_bp_s* h)
{
    const int N = h->g.numberOfPixels, P = h->g.numberOfParallelProjections, D = h->g.numberOfParallelDetectors;
    const double scale = (double)h->lut.scale;
    for (int a = 0; a < P; a++) {
        const double c = h->lut.cosT[a], sn = h->lut.sinT[a];
        if (std::max(std::fabs(c), std::fabs(sn)) * scale > 1.0) return;
    }
    const int PW = N + 2 * kAdjPad;
    const double c0 = (N - 1) * 0.5;
    const auto inside = mask_intervals(N, h->fuse_mask);
    std::vector<AdjAngle> cls[2];
    std::vector<int2> rows((size_t)P * N);
    std::vector<int> nb(P), dm(P);
    for (int a = 0; a < P; a++) {
        const double c = h->lut.cosT[a], sn = h->lut.sinT[a];
        const int k = std::fabs(c) >= std::fabs(sn) ? 0 : 1;
        const double cA = k ? sn : c, sA = k ? c : sn;
        int m = 0;
        for (int r = 0; r < N; r++) {
            const double rho = (r - c0) * (sA / cA);
            const double rd = std::floor(rho + 0.5);
            const int delta = -(int)rd;
            rows[(size_t)a * N + r] = make_int2((r * PW + kAdjPad + delta) * 4, delta * 8);
            m = std::max(m, std::abs(delta));
        }
        dm[a] = m;
        nb[a] = ceil_div(N + 2 * m, 64);
        cls[k].push_back(AdjAngle{a, k, (float)cA, -m, nb[a]});
    }
    int nbmax = 0;
    for (int a = 0; a < P; a++) nbmax = std::max(nbmax, nb[a]);
    // a row's band records must fit the reduce's LDS; 224 bands are at most 14336
    // pixels, so that a padded group of four images stays below 2^32 bytes, the
    // range of the path kernel's offsets
    if ((size_t)nbmax * kAdjRec * sizeof(float) > kMaxLds) return;
    static_assert(kMaxLds / (kAdjRec * sizeof(float)) * 64 * (kMaxLds / (kAdjRec * sizeof(float)) * 64 + 2 * kAdjPad) * 16 <
                      (size_t)1 << 32, "four padded images within 32-bit offsets");
    // rows of each band whose path segment meets the mask (one pixel of
    // margin); every row in between must stay inside the padded row
    std::vector<int2> bands((size_t)P * nbmax, make_int2(1, 0));
    for (int a = 0; a < P; a++)
        for (int b = 0; b < nb[a]; b++) {
            const int J0 = -dm[a] + 64 * b;
            int first = -1, last = -2;
            for (int r = 0; r < N; r++) {
                const int lo = inside[(size_t)r].first - 1, hi = inside[(size_t)r].second + 1;
                if (inside[(size_t)r].first > inside[(size_t)r].second) continue;
                const int x0 = rows[(size_t)a * N + r].y / 8 + J0;
                if (x0 + 63 < lo || x0 > hi) continue;
                if (first < 0) first = r;
                last = r;
            }
            if (first < 0) continue;
            for (int r = first; r <= last; r++) {
                const int x0 = rows[(size_t)a * N + r].y / 8 + J0;
                if (x0 < -kAdjPad || x0 + 63 >= N + kAdjPad) return;   // would leave the padded row: keep the gather adjoint
            }
            bands[(size_t)a * nbmax + b] = make_int2(first, last);
        }
    // sorted angle list: class A, then class B, each padded to whole workgroups
    std::vector<AdjAngle> list;
    for (int k = 0; k < 2; k++) {
        list.insert(list.end(), cls[k].begin(), cls[k].end());
        while (list.size() % kAdjWavesPerGroup) list.push_back(AdjAngle{-1, 0, 0.0f, 0, 0});
    }
    AdjParams q{};
    q.N = N;
    q.P = P;
    q.D = D;
    q.cI = (int)(D * 0.5);
    q.PW = PW;
    q.nbmax = nbmax;
    q.npos = (int)list.size();
    q.scale = h->lut.scale;
    q.center = h->lut.center;
    q.c0 = c0;
    q.outmul = h->lut.norm;
    q.img_stride = (long)N * PW;
    h->adj = q;
    h->adj_groups = (int)list.size() / kAdjWavesPerGroup;
    h->adj_angles.resize(list.size());
    h->adj_angles.upload(list);
    h->adj_rows.resize(rows.size());
    h->adj_rows.upload(rows);
    h->adj_bands.resize(bands.size());
    h->adj_bands.upload(bands);
    h->adj_nb.resize(nb.size());
    h->adj_nb.upload(nb);
    h->adj_imgA.resize((size_t)kAdjPlaces * q.img_stride);
    h->adj_imgB.resize((size_t)kAdjPlaces * q.img_stride);
    // the padding columns stay zero: pad kernels write only the N x N interior
    RISA_HIP_CHECK(hipMemset(h->adj_imgA.ptr, 0, h->adj_imgA.count * sizeof(float)));
    RISA_HIP_CHECK(hipMemset(h->adj_imgB.ptr, 0, h->adj_imgB.count * sizeof(float)));
    h->adj_partial.resize((size_t)kAdjSlices * P * nbmax * kAdjRec);
    size_t tiles = 0;
    for (int v = 0; v < kNumVariants; v++)
        tiles = std::max(tiles, (size_t)ceil_div(N, kVariants[v].tx) * ceil_div(N, kVariants[v].ty));
    h->adj_T.resize(tiles * P);
    h->adj_coord.resize(N);
    RISA_HIP_CHECK(hipDeviceSynchronize());
    h->adj_path = true;
}

extern "C" int risa_hip_bp_create(const risa_geom* g, int device, risa_bp_t* out)
{
    return guarded("risa_hip_bp_create", [&] {
        if (!g || !out) fail(RISA_ERR_ARG, "null argument");
        check_geom(g, false, true);
        DeviceGuard dg(device);
        auto h = new risa_bp_s();
        try {
            h->device = device;
            h->g = *g;
            h->lut = bp_lut(*g);
            h->cosT.resize(h->lut.cosT.size());
            h->cosT.upload(h->lut.cosT);
            h->sinT.resize(h->lut.sinT.size());
            h->sinT.upload(h->lut.sinT);
            h->fuse_mask = g->fusedMasking && !g->normalization;
            // until a variant is set or timed: the first one whose staging holds
            // a window (variant 0 up to 46 detectors per pixel, some up to 63)
            for (int v = kNumVariants - 1; v >= 0; v--) {
                const int W = window_entries(kVariants[v].tx, kVariants[v].ty, h->lut.scale);
                if (kVariants[v].stages(W) && tile_lds(1, W, kVariants[v].sb) * kVariants[v].q <= kMaxLds) h->variant = v;
            }
            // run-call scratch, sized here so run calls allocate nothing
            const size_t plane = (size_t)g->numberOfParallelProjections * g->numberOfParallelDetectors;
            h->x4.resize((size_t)kF16StageGroups * plane);
            setup_adjoint(h);
            h->imgT.resize((size_t)g->numberOfPixels * g->numberOfPixels);   // the gather adjoint's transpose
            // heaviest-first dispatch tables of every tile shape
            std::vector<int> orders;
            for (int v = 0; v < kNumVariants + kNumF16Variants; v++) {
                const int tx = v < kNumVariants ? kVariants[v].tx : kF16Variants[v - kNumVariants].tx;
                const int ty = v < kNumVariants ? kVariants[v].ty : kF16Variants[v - kNumVariants].ty;
                const std::vector<int> o = dispatch_order(make_params(h, tx, ty), tx, ty, h->fuse_mask);
                h->order_off.push_back(o.empty() ? -1L : (long)orders.size());
                orders.insert(orders.end(), o.begin(), o.end());
            }
            if (!orders.empty()) {
                h->tile_order.resize(orders.size());
                h->tile_order.upload(orders);
            }
        } catch (...) {
            delete h;
            throw;
        }
        *out = h;
    });
}

// bp_work's order for a launch whose tile shape's tables lie at `off` (-1: none,
// the tiles no multiple of 8).  Whole slice groups go to XCDs where their
// number divides; a single group, or a number that does not, takes its
// heaviest tiles first over the whole chip instead: ranges of tiles per XCD
// leave the XCDs of the image's corners idle early, and a row-major or
// Morton order ends on full tiles.  32 slices of 512^2 x 1000 on the matrix
// cores, two launches in flight: 450 us, 472 with ranges (256 frames 4.14 ms,
// 4.35); one slice of 384^2 x 360 17.6 / 23.2 us, of 640^2 x 720 55 / 63; three
// groups of 2 slices of 512^2 x 1000 199 us, 204 in tile order.
static void set_dispatch(risa_bp_t h, BpParams& p, long off, dim3 grid)
{
    p.order = off >= 0 ? h->tile_order.ptr + off : nullptr;
    p.xg = xcd_groups(grid.x, grid.y);
    if (p.order && (grid.y == 1 || !p.xg)) p.xg = 2;
}

// Slice k of the call is sino(k) -> img(k); launches of up to kBpSlices
// slices (a multiple of every variant's slices per workgroup).
template <class SinoAt, class ImgAt>
static void launch_linear_at(risa_bp_t h, int variant, SinoAt sino, ImgAt img, int slices, hipStream_t s)
{
    const BpVariant& v = kVariants[variant];
    BpParams p = make_params(h, v.tx, v.ty);
    if (!v.stages(p.W)) fail(RISA_ERR_UNSUPPORTED, "backprojection window exceeds the tile's staging");
    p.AE = chunk_angles(v.threads(), v.e, v.amax, p.W, v.sb, v.q);
    if (v.q > 1) {   // a group's chunks of about the same length
        const int len = ceil_div(p.P, v.q);
        p.AE = ceil_div(len, ceil_div(len, p.AE));
    }
    const size_t lds = std::max(v.q * tile_lds(p.AE, p.W, v.sb),
                                sizeof(float) * (v.q - 1) * v.ppt * v.sb * v.threads());
    if (lds > kMaxLds) fail(RISA_ERR_UNSUPPORTED, "backprojection tile needs %zu B of LDS", lds);
    static_assert(kBpSlices % 4 == 0, "launch chunks hold whole slice groups");
    for (int k0 = 0; k0 < slices; k0 += kBpSlices) {
        const int n = std::min(kBpSlices, slices - k0);
        BpSlices L{};
        for (int k = 0; k < n; k++) {
            L.sino[k] = sino(k0 + k);
            L.img[k] = img(k0 + k);
            if (!L.sino[k] || !L.img[k]) fail(RISA_ERR_ARG, "null slice pointer");
        }
        dim3 grid(p.tilesX * ceil_div(p.N, v.ty), ceil_div(n, v.sb));
        set_dispatch(h, p, h->order_off[(size_t)variant], grid);
        hipLaunchKernelGGL(v.fn, grid, dim3(v.q * v.threads()), lds, s, L, h->cosT.ptr, h->sinT.ptr, n, p);
        check_launch("bp_linear_kernel");
    }
}
static void launch_linear(risa_bp_t h, int variant, const float* sino, float* img, int slices, hipStream_t s)
{
    const size_t ns = (size_t)h->g.numberOfParallelProjections * h->g.numberOfParallelDetectors;
    const size_t ni = (size_t)h->g.numberOfPixels * h->g.numberOfPixels;
    launch_linear_at(
        h, variant, [&](int k) { return sino + (size_t)k * ns; }, [&](int k) { return img + (size_t)k * ni; }, slices,
        s);
}

extern "C" int risa_hip_bp_run(risa_bp_t h, const float* sino, float* img, void* stream)
{
    return guarded("risa_hip_bp_run", [&] {
        if (!h || !sino || !img) fail(RISA_ERR_ARG, "null argument");
        hipStream_t s = as_stream(stream);
        if (h->g.useTextureMemory || h->g.interpolationType == 1) {
            BpParams p = make_params(h, 16, 16);
            dim3 grid(ceil_div(p.N, 16), ceil_div(p.N, 16));
            hipLaunchKernelGGL(bp_nearest_kernel, grid, dim3(16, 16), 0, s, sino, img, h->cosT.ptr, h->sinT.ptr, p,
                               h->g.useTextureMemory ? 1 : 0);
            check_launch("bp_nearest_kernel");
            return;
        }
        launch_linear(h, h->variant, sino, img, 1, s);
    });
}

extern "C" int risa_hip_bp_run_batch(risa_bp_t h, const float* sino, int slices, float* img, void* stream)
{
    return guarded("risa_hip_bp_run_batch", [&] {
        if (!h || !sino || !img || slices < 0) fail(RISA_ERR_ARG, "bad argument");
        if (h->g.useTextureMemory || h->g.interpolationType == 1)
            fail(RISA_ERR_UNSUPPORTED, "batched backprojection is linear interpolation only");
        if (slices) launch_linear(h, h->variant, sino, img, slices, as_stream(stream));
    });
}

extern "C" int risa_hip_bp_run_list(risa_bp_t h, const float* const* sino, int slices, float* const* img,
                                    void* stream)
{
    return guarded("risa_hip_bp_run_list", [&] {
        if (!h || !sino || !img || slices < 0) fail(RISA_ERR_ARG, "bad argument");
        if (h->g.useTextureMemory || h->g.interpolationType == 1)
            fail(RISA_ERR_UNSUPPORTED, "batched backprojection is linear interpolation only");
        if (slices)
            launch_linear_at(
                h, h->variant, [&](int k) { return sino[k]; }, [&](int k) { return img[k]; }, slices,
                as_stream(stream));
    });
}

static void launch_f16x4(risa_bp_t h, int variant, const uint2* sino, float in_scale, int slices, float* img,
                         hipStream_t s)
{
    const BpF16Variant& v = kF16Variants[variant];
    BpParams p = make_params(h, v.tx, v.ty);
    p.out_scale = 1.0f / in_scale;
    const int threads = v.tx * v.ty / v.ppt;
    // per group an LDS plane of two chunks of E * threads entries
    if (p.W > v.e * threads) fail(RISA_ERR_UNSUPPORTED, "backprojection window exceeds the tile's staging");
    p.AE = std::max(1, std::min(v.amax, v.e * threads / p.W));
    if (v.q > 1) {   // a group's chunks of about the same length
        const int len = ceil_div(p.P, v.q);
        p.AE = ceil_div(len, ceil_div(len, p.AE));
    }
    const size_t lds = std::max(v.q * f16_lds(v.g, v.e, threads, p.AE),
                                sizeof(float) * (v.q - 1) * v.ppt * kF16Group * v.g * threads);
    if (lds > (v.q > 1 ? kMaxLds / 64 * 80 : kMaxLds)) fail(RISA_ERR_UNSUPPORTED, "backprojection tile needs %zu B of LDS", lds);
    dim3 grid(p.tilesX * ceil_div(p.N, v.ty), ceil_div(ceil_div(slices, kF16Group), v.g));
    set_dispatch(h, p, h->order_off[(size_t)(kNumVariants + variant)], grid);
    hipLaunchKernelGGL(v.fn, grid, dim3(v.q * threads), lds, s, sino, img, h->cosT.ptr, h->sinT.ptr, slices, p);
    check_launch("bp_linear_f16_kernel");
}

extern "C" int risa_hip_bp_run_f16x4(risa_bp_t h, const uint16_t* sino_x4, float in_scale, int slices, float* img,
                                     void* stream)
{
    return guarded("risa_hip_bp_run_f16x4", [&] {
        if (!h || !sino_x4 || !img || slices < 0 || !(in_scale > 0)) fail(RISA_ERR_ARG, "bad argument");
        if (reinterpret_cast<uintptr_t>(sino_x4) % 8) fail(RISA_ERR_ARG, "x4 sinogram must be 8-byte aligned");
        if (slices) launch_f16x4(h, h->variant_f16, reinterpret_cast<const uint2*>(sino_x4), in_scale, slices, img,
                                 as_stream(stream));
    });
}

extern "C" int risa_hip_bp_run_f16(risa_bp_t h, const uint16_t* sino, float in_scale, int slices, float* img,
                                   void* stream)
{
    return guarded("risa_hip_bp_run_f16", [&] {
        if (!h || !sino || !img || slices < 0 || !(in_scale > 0)) fail(RISA_ERR_ARG, "bad argument");
        if (!slices) return;
        hipStream_t s = as_stream(stream);
        const long plane = (long)h->g.numberOfParallelProjections * h->g.numberOfParallelDetectors;
        // passes of up to kF16StageGroups * 4 slices through the staging
        // buffer; stream order keeps a pass's conversion behind the previous
        // pass's backprojection
        const int per = kF16StageGroups * kF16Group;
        for (int s0 = 0; s0 < slices; s0 += per) {
            const int n = std::min(per, slices - s0);
            hipLaunchKernelGGL(f16_to_x4_kernel, dim3(1024), dim3(256), 0, s, sino + (size_t)s0 * plane, h->x4.ptr, n,
                               plane);
            check_launch("f16_to_x4_kernel");
            launch_f16x4(h, h->variant_f16, h->x4.ptr, in_scale, n, img + (size_t)s0 * h->g.numberOfPixels *
                         h->g.numberOfPixels, s);
        }
    });
}

// ------------------------------------------ FP32 split backprojection --
// Used by the chain for groups of many frames (chain.hip); its sums are
// rounded otherwise than bp_linear_kernel's, and no less exact.
struct SplitShape {
    int tx, ty, amax, variant;   // variant: an FP32 variant of the same tile shape (its dispatch order)
    void (*fn[2])(const unsigned*, float*, const float*, const float*, int, BpParams);   // up to 16 and 32 slices
};
static const SplitShape kSplitShapes[] = {
    {32, 32, 8, 0, {bp_split_kernel<32, 32, 1>, bp_split_kernel<32, 32, 2>}},
    {32, 16, 4, 1, {bp_split_kernel<32, 16, 1>, bp_split_kernel<32, 16, 2>}},
    {16, 16, 4, 2, {bp_split_kernel<16, 16, 1>, bp_split_kernel<16, 16, 2>}},
};
constexpr int kNumSplitShapes = sizeof(kSplitShapes) / sizeof(kSplitShapes[0]);
constexpr int kMaxSplitLds = 160 * 1024;   // a gfx950 workgroup's LDS
constexpr int kMaxPackAngles = 65535;      // the packing kernels take one grid row per angle

// Angles of a shape's chunk: the shape's most, or half as often as its LDS asks.
static int split_angles(int shape, int W)
{
    int ae = kSplitShapes[shape].amax;
    while (ae > 4 && split_lds(ae, W) > kMaxSplitLds) ae /= 2;
    return ae;
}

// What a workgroup of `shape` stages at a detector scale, for checks on the
// host: window samples W, angles per chunk, rows copied per angle, bytes of a
// row, bytes between angles, bytes of a buffer, LDS bytes.
extern "C" int risa_bp_split_layout(int shape, float scale, int layout[7])
{
    return guarded("risa_bp_split_layout", [&] {
        if (shape < 0 || shape >= kNumSplitShapes || !(scale > 0.0f) || scale > kSplitMaxScale || !layout)
            fail(RISA_ERR_ARG, "bad argument");
        const int W = window_entries(kSplitShapes[shape].tx, kSplitShapes[shape].ty, scale), ae = split_angles(shape, W);
        const int v[7] = {W, ae, split_staged(W), kSplitRow, split_pitch(W), split_buffer(ae, W), split_lds(ae, W)};
        std::copy(v, v + 7, layout);
    });
}

// Bytes of the packed sinograms of one launch (32 slices); 0 where the
// geometry is outside what the kernel takes.
extern "C" size_t risa_bp_split_bytes(risa_bp_t h)
{
    const risa_geom& g = h->g;
    if (g.useTextureMemory || g.interpolationType == 1 || h->lut.scale > kSplitMaxScale ||
        g.numberOfParallelProjections > kMaxPackAngles)
        return 0;
    return (size_t)g.numberOfParallelProjections * split_rows(g.numberOfParallelDetectors) * kSplitRow;
}

// Up to 32 sinograms [slices][P][D] -> images [slices][N][N] with tile shape
// `shape`; |value * scale| must stay within the FP16 range.  `packed`:
// risa_bp_split_bytes of scratch, 16-byte aligned.
extern "C" int risa_bp_run_split(risa_bp_t h, int shape, const float* sino, float scale, int slices, void* packed, float* img,
                      hipStream_t s)
{
    return guarded("risa_bp_run_split", [&] {
        if (shape < 0 || shape >= kNumSplitShapes || slices < 1 || slices > kSplitSlices || !(scale > 0.0f))
            fail(RISA_ERR_ARG, "bad argument");
        if (risa_bp_split_bytes(h) == 0) fail(RISA_ERR_UNSUPPORTED, "geometry outside the split backprojector's range");
        const SplitShape& v = kSplitShapes[shape];
        BpParams p = make_params(h, v.tx, v.ty);
        p.out_scale = 1.0f / scale;
        p.AE = split_angles(shape, p.W);
        const int lds = split_lds(p.AE, p.W);
        if (lds > kMaxSplitLds) fail(RISA_ERR_UNSUPPORTED, "backprojection tile needs %d B of LDS", lds);
        dim3 grid(p.tilesX * ceil_div(p.N, v.ty), 1);
        set_dispatch(h, p, h->order_off[(size_t)v.variant], grid);
        unsigned* pk = reinterpret_cast<unsigned*>(packed);
        hipLaunchKernelGGL(split_pack_kernel, dim3(ceil_div(split_rows(p.D) - 2, 32), p.P), dim3(256), 0, s, sino,
                           slices, p.P, p.D, scale, pk);
        check_launch("split_pack_kernel");
        hipLaunchKernelGGL(v.fn[slices > kSplitSlices / 2], grid, dim3(v.tx * v.ty), lds, s, pk, img, h->cosT.ptr,
                           h->sinT.ptr, slices, p);
        check_launch("bp_split_kernel");
    });
}

// Times the split shapes at 32 slices against the handle's FP32 variant on
// the same launch: `shape` gets the fastest one, cost[0] and cost[1] what its
// launches of up to 16 and up to 32 slices take, in slices of the variant (whose
// time is about proportional).
extern "C" int risa_bp_tune_split(risa_bp_t h, hipStream_t s, int* shape, float cost[2])
{
    return guarded("risa_bp_tune_split", [&] {
        DeviceGuard dg(h->device);
        const size_t ns = (size_t)h->g.numberOfParallelProjections * h->g.numberOfParallelDetectors;
        const size_t ni = (size_t)h->g.numberOfPixels * h->g.numberOfPixels;
        DeviceBuffer<float> sino(ns * kSplitSlices), img(ni * kSplitSlices);
        DeviceBuffer<char> packed(risa_bp_split_bytes(h));
        // values that toggle the multipliers as real ones do
        hipLaunchKernelGGL(tune_fill_kernel, dim3(1024), dim3(256), 0, s, sino.ptr, (long)sino.count);
        check_launch("tune_fill_kernel");
        struct Events {
            hipEvent_t a = nullptr, b = nullptr;
            ~Events()
            {
                if (a) (void)hipEventDestroy(a);
                if (b) (void)hipEventDestroy(b);
            }
        } ev;
        RISA_HIP_CHECK(hipEventCreate(&ev.a));
        RISA_HIP_CHECK(hipEventCreate(&ev.b));
        auto time_it = [&](auto&& launch) {
            launch();
            RISA_HIP_CHECK(hipEventRecord(ev.a, s));
            for (int it = 0; it < 5; it++) launch();
            RISA_HIP_CHECK(hipEventRecord(ev.b, s));
            RISA_HIP_CHECK(hipEventSynchronize(ev.b));
            float ms = 0;
            RISA_HIP_CHECK(hipEventElapsedTime(&ms, ev.a, ev.b));
            return ms;
        };
        auto time_split = [&](int v, int slices) {
            return time_it([&] {
                if (risa_bp_run_split(h, v, sino.ptr, 1024.0f, slices, packed.ptr, img.ptr, s) != RISA_OK)
                    fail(RISA_ERR_HIP, "%s", risa_last_error());
            });
        };
        float plain = 1e30f, best = 1e30f, half = 1e30f;
        *shape = 0;
        for (int round = 0; round < 2; round++) {
            plain = std::min(plain, time_it([&] { launch_linear(h, h->variant, sino.ptr, img.ptr, kSplitSlices, s); }));
            for (int v = 0; v < kNumSplitShapes; v++) {
                const float ms = time_split(v, kSplitSlices);
                if (ms < best) {
                    best = ms;
                    *shape = v;
                }
            }
        }
        for (int round = 0; round < 2; round++) half = std::min(half, time_split(*shape, kSplitSlices / 2));
        cost[0] = kSplitSlices * half / plain;
        cost[1] = kSplitSlices * best / plain;
    });
}

static void autotune(risa_bp_t h, int s32, int s16, hipStream_t s, int max_sb = 1, bool keep_tile = false,
                     int max_q = INT_MAX);

// -------------------------------- FP16 backprojection of 64 slices at once --
// Used by the mixed chain for groups of many frames (chain.hip), in place of an
// FP16 variant whose results it has bit for bit.
static bool f16_packable(risa_bp_t h)
{
    const risa_geom& g = h->g;
    const BpF16Variant& v = kF16Variants[h->variant_f16];
    return !g.useTextureMemory && g.interpolationType != 1 && h->lut.scale <= kSplitMaxScale &&
           g.numberOfParallelProjections <= kMaxPackAngles && v.tx == 16 && v.ty == 16;
}

// Bytes of packed samples for 64 slices, or 0 where the handle's geometry or
// its FP16 variant (another tile than 16 x 16, or shared angles) has no
// counterpart there.
extern "C" size_t risa_bp_f16_pack_bytes(risa_bp_t h)
{
    const risa_geom& g = h->g;
    if (!f16_packable(h) || kF16Variants[h->variant_f16].q != 1) return 0;
    return (size_t)g.numberOfParallelProjections * pack_rows(g.numberOfParallelDetectors) * kPackSlices * 4;
}

// Up to 64 slices of the x4 layout -> images; `packed`: risa_bp_f16_pack_bytes
// of scratch, 16-byte aligned.
extern "C" int risa_bp_run_f16_packed(risa_bp_t h, const uint16_t* sino_x4, float in_scale, int slices, void* packed,
                                      float* img, hipStream_t s)
{
    return guarded("risa_bp_run_f16_packed", [&] {
        if (slices < 1 || slices > kPackSlices || !(in_scale > 0)) fail(RISA_ERR_ARG, "bad argument");
        if (risa_bp_f16_pack_bytes(h) == 0) fail(RISA_ERR_UNSUPPORTED, "no packed form of this FP16 variant");
        constexpr int kTile = 32, kParts = 4;
        BpParams p = make_params(h, kTile, kTile);
        p.out_scale = 1.0f / in_scale;
        p.AE = 4;
        while (p.AE > 1 && pack_lds(p.AE, p.W, kParts) > kMaxSplitLds) p.AE /= 2;
        const int lds = pack_lds(p.AE, p.W, kParts);
        if (lds > kMaxSplitLds) fail(RISA_ERR_UNSUPPORTED, "backprojection tile needs %d B of LDS", lds);
        dim3 grid(p.tilesX * ceil_div(p.N, kTile), 1);
        // ranges of tiles per XCD: 705 us, 720 heaviest first over the chip
        p.xg = xcd_groups(grid.x, 1);
        const long off = h->order_off[0];   // the first FP32 variant has this tile
        p.order = p.xg && off >= 0 ? h->tile_order.ptr + off : nullptr;
        const uint2* x4 = reinterpret_cast<const uint2*>(sino_x4);
        uint4* pk = reinterpret_cast<uint4*>(packed);
        hipLaunchKernelGGL(f16_pack_kernel, dim3(ceil_div(pack_rows(p.D), 64), p.P), dim3(256), 0, s, x4,
                           ceil_div(slices, kF16Group), p.P, p.D, pk);
        check_launch("f16_pack_kernel");
        hipLaunchKernelGGL((bp_f16_mfma_kernel<kTile, kTile, 4>), grid, dim3(kTile * kTile), lds, s, pk, x4, img, h->cosT.ptr, h->sinT.ptr, slices, p);
        check_launch("bp_f16_mfma_kernel");
    });
}

// Times it at 64 slices against the handle's FP16 variant, where that has a
// 16 x 16 tile: `min_slices` is the batch from which it is the faster one (its
// cost does not depend on the slices up to 64), or more than 64 if never.  If it
// is, a variant with shared angles gives way to the fastest one of the same tile
// without at `slices` slices, whose bits the packed kernel has, for the batches
// below.
extern "C" int risa_bp_tune_f16_packed(risa_bp_t h, hipStream_t s, int slices, int* min_slices)
{
    return guarded("risa_bp_tune_f16_packed", [&] {
        *min_slices = kPackSlices + 1;
        if (!f16_packable(h)) return;
        DeviceGuard dg(h->device);
        const size_t ns = (size_t)h->g.numberOfParallelProjections * h->g.numberOfParallelDetectors;
        const size_t ni = (size_t)h->g.numberOfPixels * h->g.numberOfPixels;
        const int own = h->variant_f16;
        if (kF16Variants[own].q != 1) autotune(h, 0, slices, s, 1, true, 1);
        const int whole = h->variant_f16;
        DeviceBuffer<uint16_t> sino(ns * kPackSlices);
        DeviceBuffer<float> img(ni * kPackSlices);
        DeviceBuffer<char> packed(risa_bp_f16_pack_bytes(h));
        hipLaunchKernelGGL(tune_fill_f16_kernel, dim3(1024), dim3(256), 0, s, sino.ptr, (long)sino.count);
        check_launch("tune_fill_f16_kernel");
        hipEvent_t ev[2] = {};
        auto destroy = [&] {
            for (hipEvent_t e : ev)
                if (e) (void)hipEventDestroy(e);
        };
        try {
            for (hipEvent_t& e : ev) RISA_HIP_CHECK(hipEventCreate(&e));
            auto time_it = [&](auto&& launch) {
                launch();
                RISA_HIP_CHECK(hipEventRecord(ev[0], s));
                for (int it = 0; it < 5; it++) launch();
                RISA_HIP_CHECK(hipEventRecord(ev[1], s));
                RISA_HIP_CHECK(hipEventSynchronize(ev[1]));
                float ms = 0;
                RISA_HIP_CHECK(hipEventElapsedTime(&ms, ev[0], ev[1]));
                return ms;
            };
            float plain = 1e30f, best = 1e30f;
            for (int round = 0; round < 2; round++) {
                plain = std::min(plain, time_it([&] {
                                     launch_f16x4(h, own, reinterpret_cast<const uint2*>(sino.ptr), 1.0f, kPackSlices,
                                                  img.ptr, s);
                                 }));
                best = std::min(best, time_it([&] {
                                    if (risa_bp_run_f16_packed(h, sino.ptr, 1.0f, kPackSlices, packed.ptr, img.ptr, s) !=
                                        RISA_OK)
                                        fail(RISA_ERR_HIP, "%s", risa_last_error());
                                }));
            }
            *min_slices = 1 + (int)(kPackSlices * best / plain);
        } catch (...) {
            destroy();
            h->variant_f16 = own;
            throw;
        }
        destroy();
        h->variant_f16 = *min_slices <= kPackSlices ? whole : own;
    });
}

// The gather adjoint (bp_adjoint_kernel) of one slice: geometries the
// sheared-path kernel does not cover (scale > 1).
static void adjoint_gather(risa_bp_t h, const float* img, float* sino, hipStream_t s)
{
    // the transpose of the FP32 linear kernel the handle runs: same tile shape
    const BpVariant& v = kVariants[h->variant];
    BpParams p = make_params(h, v.tx, v.ty);
    const int tilesY = ceil_div(p.N, v.ty);
    int ltx = 0, lty = 0;
    while ((1 << ltx) < v.tx) ltx++;
    while ((1 << lty) < v.ty) lty++;
    if ((1 << ltx) != v.tx || (1 << lty) != v.ty) fail(RISA_ERR_UNSUPPORTED, "adjoint needs power-of-two tile edges");
    // a line's span for kAdjK detectors: (kAdjK + 2) / (|cos or sin| scale)
    // pixels with |cos or sin| >= 1/sqrt(2), plus slack and rounding
    const int cap = std::min(p.N, (int)std::ceil((kAdjK + 2) * 1.41422 / p.scale) + 6);
    const size_t lds = (size_t)p.tilesX * tilesY * 8 + (size_t)p.N * 8 + kAdjWaves * kAdjK * sizeof(float) +
                       (size_t)kAdjWaves * cap * 12;
    if (lds > kMaxLds) fail(RISA_ERR_UNSUPPORTED, "adjoint: its tables need %zu B of LDS", lds);
    hipLaunchKernelGGL(transpose_kernel, dim3(ceil_div(p.N, 32), ceil_div(p.N, 32)), dim3(32, 8), 0, s, img,
                       h->imgT.ptr, p.N);
    check_launch("transpose_kernel");
    dim3 grid(ceil_div(p.D, kAdjK), p.P);
    hipLaunchKernelGGL(bp_adjoint_kernel, grid, dim3(64 * kAdjWaves), lds, s, img, h->imgT.ptr, sino, h->cosT.ptr,
                       h->sinT.ptr, p, ltx, lty, tilesY, cap);
    check_launch("bp_adjoint_kernel");
}

// `slices` images [N][N] -> sinograms [P][D]: passes of up to kAdjSlices
// slices through the handle's padded copies and partial windows (allocated
// at create; stream order keeps a pass behind the previous one).
// log2 of a power-of-two tile edge
static int ilog2(int v)
{
    int l = 0;
    while ((1 << l) < v) l++;
    if ((1 << l) != v) fail(RISA_ERR_UNSUPPORTED, "tile edge %d is not a power of two", v);
    return l;
}

static void adjoint_run(risa_bp_t h, const float* img, int slices, float* sino, hipStream_t s)
{
    const int N = h->g.numberOfPixels;
    const long P = h->g.numberOfParallelProjections, D = h->g.numberOfParallelDetectors;
    if (!h->adj_path || h->adj_gather) {
        for (int i = 0; i < slices; i++) adjoint_gather(h, img + (size_t)i * N * N, sino + (size_t)i * P * D, s);
        return;
    }
    AdjParams q = h->adj;
    // the forward's tile grid of the variant in use, and its tile origins
    const BpVariant& v = kVariants[h->variant];
    q.lgTX = ilog2(v.tx);
    q.lgTY = ilog2(v.ty);
    q.tilesX = ceil_div(N, v.tx);
    q.tilesY = ceil_div(N, v.ty);
    const long work = std::max((long)q.tilesX * q.tilesY * P, (long)N);
    hipLaunchKernelGGL(adj_tile_origin_kernel, dim3((unsigned)ceil_div(work, 256L)), dim3(256), 0, s, h->cosT.ptr,
                       h->sinT.ptr, q, h->adj_T.ptr, h->adj_coord.ptr);
    check_launch("adj_tile_origin_kernel");
    for (int s0 = 0; s0 < slices; s0 += kAdjSlices) {
        const int n = std::min(kAdjSlices, slices - s0);
        // 3 left over run as a group of 4
        q.quads = (n + 1) / 4;
        q.tail = n % 4 == 3 ? 0 : n % 4;
        const unsigned groups = (unsigned)(q.quads + (q.tail ? 1 : 0));
        hipLaunchKernelGGL(adj_pad_kernel, dim3(ceil_div(N, 32), ceil_div(N, 32), groups), dim3(32, 8), 0, s,
                           img + (size_t)s0 * N * N, n, h->adj_imgA.ptr, h->adj_imgB.ptr, N, q.PW,
                           h->fuse_mask ? 1 : 0, h->lut.center, q.img_stride, q.quads, q.tail);
        check_launch("adj_pad_kernel");
        const auto path = q.tail == 0   ? bp_adjoint_path_kernel<true, 0>
                          : q.tail == 1 ? (q.quads ? bp_adjoint_path_kernel<true, 1> : bp_adjoint_path_kernel<false, 1>)
                                        : (q.quads ? bp_adjoint_path_kernel<true, 2> : bp_adjoint_path_kernel<false, 2>);
        hipLaunchKernelGGL(path, dim3(h->adj_groups, q.nbmax, groups), dim3(64 * kAdjWavesPerGroup), 0, s,
                           h->adj_imgA.ptr, h->adj_imgB.ptr, h->adj_partial.ptr, h->adj_angles.ptr, h->adj_bands.ptr,
                           h->adj_rows.ptr, h->adj_coord.ptr, h->adj_T.ptr, h->cosT.ptr, h->sinT.ptr, n, q);
        check_launch("bp_adjoint_path_kernel");
        hipLaunchKernelGGL(adj_reduce_kernel, dim3(P, n), dim3(256), (size_t)q.nbmax * kAdjRec * sizeof(float), s,
                           h->adj_partial.ptr, h->adj_nb.ptr, sino + (size_t)s0 * P * D, q);
        check_launch("adj_reduce_kernel");
    }
}

extern "C" int risa_hip_bp_adjoint_run(risa_bp_t h, const float* img, float* sino, void* stream)
{
    return guarded("risa_hip_bp_adjoint_run", [&] {
        if (!h || !img || !sino) fail(RISA_ERR_ARG, "null argument");
        adjoint_run(h, img, 1, sino, as_stream(stream));
    });
}

extern "C" int risa_hip_bp_adjoint_run_batch(risa_bp_t h, const float* img, int slices, float* sino, void* stream)
{
    return guarded("risa_hip_bp_adjoint_run_batch", [&] {
        if (!h || !img || !sino || slices < 0) fail(RISA_ERR_ARG, "bad argument");
        if (slices) adjoint_run(h, img, slices, sino, as_stream(stream));
    });
}

extern "C" int risa_hip_bp_adjoint_method(risa_bp_t h, int method)
{
    return guarded("risa_hip_bp_adjoint_method", [&] {
        if (!h) fail(RISA_ERR_ARG, "null handle");
        if (method != 0 && method != 1) fail(RISA_ERR_ARG, "adjoint method must be 0 or 1");
        h->adj_gather = method == 1;
    });
}

extern "C" int risa_hip_bp_set_variant(risa_bp_t h, int variant)
{
    return guarded("risa_hip_bp_set_variant", [&] {
        if (!h) fail(RISA_ERR_ARG, "null handle");
        // low 8 bits: FP32 variant; next 8 bits: FP16 variant
        const int v32 = variant & 0xff, v16 = (variant >> 8) & 0xff;
        if (v32 >= kNumVariants || v16 >= kNumF16Variants || variant < 0) fail(RISA_ERR_ARG, "variant out of range");
        h->variant = v32;
        h->variant_f16 = v16;
    });
}

extern "C" int risa_hip_bp_variant_shape(int f16, int variant, int shape[7])
{
    return guarded("risa_hip_bp_variant_shape", [&] {
        if (!shape || variant < 0) fail(RISA_ERR_ARG, "bad argument");
        if (f16) {
            if (variant >= kNumF16Variants) fail(RISA_ERR_ARG, "variant out of range");
            const BpF16Variant& v = kF16Variants[variant];
            const int s[7] = {v.tx, v.ty, v.ppt, v.e, v.u, v.g, v.amax};
            std::copy(s, s + 7, shape);
        } else {
            if (variant >= kNumVariants) fail(RISA_ERR_ARG, "variant out of range");
            const BpVariant& v = kVariants[variant];
            const int s[7] = {v.tx, v.ty, v.ppt, v.e, v.u, v.sb, v.amax};
            std::copy(s, s + 7, shape);
        }
    });
}

// Groups of threads that share a variant's angles (0 past the last variant).
extern "C" int risa_bp_variant_groups(int f16, int variant)
{
    if (variant < 0 || variant >= (f16 ? kNumF16Variants : kNumVariants)) return 0;
    return f16 ? kF16Variants[variant].q : kVariants[variant].q;
}

extern "C" int risa_hip_bp_get_variant(risa_bp_t h, int* variant)
{
    return guarded("risa_hip_bp_get_variant", [&] {
        if (!h || !variant) fail(RISA_ERR_ARG, "null argument");
        *variant = h->variant | (h->variant_f16 << 8);
    });
}

// Times every variant that fits the geometry with HIP events and keeps the
// fastest: FP32 variants at s32 slices per launch (the frames a caller keeps
// in flight), FP16 variants at s16 slices per launch; 0 skips a precision.
// max_sb: the FP32 variants considered take at most this many slices per
// workgroup (1 for callers that launch one slice at a time).
//
// The FP16 tile shape is picked among the variants whose angles are not shared,
// or kept (keep_tile), and the variant among those of that shape, with angles
// shared by at most max_q groups: a weight's
// FP16 rounding depends on t's distance from the tile's origin, so results move
// by up to 2e-5 (noise) from one shape to another, and by the order of the sums,
// 1e-6, within one.
static void autotune(risa_bp_t h, int s32, int s16, hipStream_t s, int max_sb, bool keep_tile, int max_q)
{
    DeviceGuard dg(h->device);
    const BpF16Variant kept = kF16Variants[h->variant_f16];
    const int N = h->g.numberOfPixels, P = h->g.numberOfParallelProjections, D = h->g.numberOfParallelDetectors;
    DeviceBuffer<float> sino((size_t)P * D * std::max(1, s32));
    DeviceBuffer<uint2> sino16((size_t)P * D * std::max(1, ceil_div(s16, kF16Group)));
    DeviceBuffer<float> img((size_t)N * N * std::max(std::max(s32, s16), 1));
    RISA_HIP_CHECK(hipMemsetAsync(sino.ptr, 0, sino.count * sizeof(float), s));
    RISA_HIP_CHECK(hipMemsetAsync(sino16.ptr, 0, sino16.count * sizeof(uint2), s));
    hipEvent_t e0, e1;
    RISA_HIP_CHECK(hipEventCreate(&e0));
    RISA_HIP_CHECK(hipEventCreate(&e1));
    auto time_it = [&](auto&& launch) {
        launch();
        RISA_HIP_CHECK(hipEventRecord(e0, s));
        for (int it = 0; it < 5; it++) launch();
        RISA_HIP_CHECK(hipEventRecord(e1, s));
        RISA_HIP_CHECK(hipEventSynchronize(e1));
        float ms = 0;
        RISA_HIP_CHECK(hipEventElapsedTime(&ms, e0, e1));
        return ms;
    };
    try {
        // two rounds over the table, each variant's best time counts: the
        // first launches of a run meet clocks still ramping up
        std::vector<float> t32(kNumVariants, 1e30f), t16(kNumF16Variants, 1e30f);
        for (int round = 0; round < 2; round++) {
            for (int v = 0; s32 > 0 && v < kNumVariants; v++) {
                if (kVariants[v].sb > max_sb) continue;
                try {
                    t32[v] = std::min(t32[v], time_it([&] { launch_linear(h, v, sino.ptr, img.ptr, s32, s); }));
                } catch (const Error& e) {
                    if (e.code != RISA_ERR_UNSUPPORTED) throw;   // this tile shape does not fit the geometry
                }
            }
            for (int v = 0; s16 > 0 && v < kNumF16Variants; v++) {
                if (keep_tile && (kF16Variants[v].tx != kept.tx || kF16Variants[v].ty != kept.ty)) continue;
                if (kF16Variants[v].q > max_q) continue;
                try {
                    t16[v] = std::min(t16[v],
                                      time_it([&] { launch_f16x4(h, v, sino16.ptr, 1.0f, s16, img.ptr, s); }));
                } catch (const Error& e) {
                    if (e.code != RISA_ERR_UNSUPPORTED) throw;
                }
            }
        }
        const auto b32 = std::min_element(t32.begin(), t32.end());
        auto b16 = std::min_element(t16.begin(), t16.end());
        if (!keep_tile) {
            int base = 0;
            for (int v = 0; v < kNumF16Variants; v++)
                if (kF16Variants[v].q == 1 && t16[v] < t16[base]) base = v;
            b16 = t16.begin() + base;
            for (int v = 0; v < kNumF16Variants; v++)
                if (kF16Variants[v].tx == kF16Variants[base].tx && kF16Variants[v].ty == kF16Variants[base].ty &&
                    t16[v] < *b16)
                    b16 = t16.begin() + v;
        }
        if (s32 > 0 && *b32 < 1e30f) h->variant = (int)(b32 - t32.begin());
        if (s16 > 0 && *b16 < 1e30f) h->variant_f16 = (int)(b16 - t16.begin());
    } catch (...) {
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        throw;
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
}

extern "C" int risa_hip_bp_autotune_slices(risa_bp_t h, int slices, void* stream)
{
    return guarded("risa_hip_bp_autotune_slices", [&] {
        if (!h || slices < 1) fail(RISA_ERR_ARG, "bad argument");
        autotune(h, slices, std::max(8, slices), as_stream(stream));
    });
}

extern "C" int risa_hip_bp_autotune_batch(risa_bp_t h, int slices, void* stream)
{
    return guarded("risa_hip_bp_autotune_batch", [&] {
        if (!h || slices < 1) fail(RISA_ERR_ARG, "bad argument");
        autotune(h, slices, 0, as_stream(stream), std::min(slices, 4));
    });
}

extern "C" int risa_hip_bp_slices_per_tile(risa_bp_t h, int* slices)
{
    return guarded("risa_hip_bp_slices_per_tile", [&] {
        if (!h || !slices) fail(RISA_ERR_ARG, "null argument");
        *slices = kVariants[h->variant].sb;
    });
}

// The fastest FP16 variant of the current one's tile shape at `slices`.
extern "C" int risa_bp_autotune_f16_tile(risa_bp_t h, int slices)
{
    return guarded("risa_bp_autotune_f16_tile", [&] {
        if (!h || slices < 1) fail(RISA_ERR_ARG, "bad argument");
        autotune(h, 0, slices, nullptr, 1, true);
    });
}

extern "C" int risa_hip_bp_autotune_f16(risa_bp_t h, int slices, void* stream)
{
    return guarded("risa_hip_bp_autotune_f16", [&] {
        if (!h || slices < 1) fail(RISA_ERR_ARG, "bad argument");
        autotune(h, 0, slices, as_stream(stream));
    });
}

extern "C" int risa_hip_bp_autotune(risa_bp_t h, void* stream)
{
    return risa_hip_bp_autotune_slices(h, 1, stream);
}

extern "C" int risa_hip_bp_destroy(risa_bp_t h)
{
    return guarded("risa_hip_bp_destroy", [&] {
        if (h) drain_device(h->device);
        delete h;
    });
}

// ---------------------------------------------------------------- Masking --
struct risa_mask_s {
    int device = 0;
    risa_geom g{};
    DeviceBuffer<float2> partial;
    int nparts = 0;
};

extern "C" int risa_hip_mask_create(const risa_geom* g, int device, risa_mask_t* out)
{
    return guarded("risa_hip_mask_create", [&] {
        if (!g || !out) fail(RISA_ERR_ARG, "null argument");
        if (g->numberOfPixels <= 0) fail(RISA_ERR_ARG, "numberOfPixels must be positive");
        DeviceGuard dg(device);
        auto h = new risa_mask_s();
        h->device = device;
        h->g = *g;
        h->nparts = std::min(256, std::max(1, ceil_div((long)g->numberOfPixels * g->numberOfPixels, 1024)));
        try {
            h->partial.resize(h->nparts);
        } catch (...) {
            delete h;
            throw;
        }
        *out = h;
    });
}

extern "C" int risa_hip_mask_run(risa_mask_t h, float* img, void* stream)
{
    return guarded("risa_hip_mask_run", [&] {
        if (!h || !img) fail(RISA_ERR_ARG, "null argument");
        hipStream_t s = as_stream(stream);
        const int N = h->g.numberOfPixels;
        const float center = (float)((N - 1.0) * 0.5);
        if (h->g.normalization) {
            hipLaunchKernelGGL(minmax_partial_kernel, dim3(h->nparts), dim3(256), 0, s, img, (long)N * N,
                               h->partial.ptr);
            check_launch("minmax_partial_kernel");
        }
        dim3 grid(ceil_div(N, 16), ceil_div(N, 16));
        hipLaunchKernelGGL(mask_apply_kernel, grid, dim3(16, 16), 0, s, img, N, center, (float)h->g.maskingValue,
                           h->g.normalization ? 1 : 0, h->partial.ptr, h->nparts);
        check_launch("mask_apply_kernel");
    });
}

extern "C" int risa_hip_mask_destroy(risa_mask_t h)
{
    return guarded("risa_hip_mask_destroy", [&] {
        if (h) drain_device(h->device);
        delete h;
    });
}

// ------------------------------------------- persistent uneven batches (C3) --
namespace risa {

struct PersistentVariant {
    int tx, ty, ppt, e, u, amax;
    void (*fn)(const BpJobDev*, const int2*, int, const float*, const float*, int*);
};
#define RISA_BPP(TX, TY, PPT, E, U, AMAX) {TX, TY, PPT, E, U, AMAX, bp_persistent_kernel<TX, TY, PPT, E, U>}
static const PersistentVariant kPersistent[] = {
    RISA_BPP(32, 32, 4, 8, 4, 64), RISA_BPP(32, 16, 2, 8, 4, 64), RISA_BPP(16, 16, 1, 4, 4, 64),
    RISA_BPP(32, 16, 4, 16, 4, 64),
};
#undef RISA_BPP
static constexpr int kNumPersistent = sizeof(kPersistent) / sizeof(kPersistent[0]);

}  // namespace risa

struct risa_bp_batched_s {
    int device = 0;
    std::vector<risa_bp_job> jobs;
    std::vector<int> lut_off;
    risa::DeviceBuffer<float> cosT, sinT;
    risa::DeviceBuffer<risa::BpJobDev> djobs;
    risa::DeviceBuffer<int2> tiles;
    risa::DeviceBuffer<int> counter;
    int ntiles = 0;
    int variant = 0;
    int grid = 0;
    size_t lds = 0;
};

// Job table and cost-sorted tile list for the current variant; refuses, before
// it changes the layout, jobs whose windows the variant cannot stage.
static void batched_layout(risa_bp_batched_s* h)
{
    const PersistentVariant& v = kPersistent[h->variant];
    std::vector<BpJobDev> dj(h->jobs.size());
    std::vector<std::pair<long, int2>> order;
    size_t lds = 0;
    const int threads = v.tx * v.ty / v.ppt;
    for (size_t i = 0; i < h->jobs.size(); i++) {
        const risa_bp_job& j = h->jobs[i];
        check_sino_size(j.P, j.D);
        BpParams p{};
        p.N = j.N; p.P = j.P; p.D = j.D;
        p.cI = (int)(j.D * 0.5);
        p.scale = (float)j.D / (float)j.N;
        p.norm = (float)(M_PI / j.P / (double)p.scale);
        p.center = (float)((j.N - 1.0) * 0.5);
        p.mask = j.mask ? 1 : 0;
        p.maskingValue = j.maskingValue;
        p.W = window_entries(v.tx, v.ty, p.scale);
        if (p.W > v.e * threads) fail(RISA_ERR_UNSUPPORTED, "job %zu: backprojection window exceeds the tile's staging", i);
        p.tilesX = ceil_div(j.N, v.tx);
        p.zx = p.zy = -1;   // the persistent kernel takes tiles from its cost-sorted list
        const int tilesY = ceil_div(j.N, v.ty);
        p.invW = 1.0f / (float)p.W;
        p.out_scale = j.dtype == RISA_F16 ? 1.0f / j.in_scale : 1.0f;
        p.AE = chunk_angles(threads, v.e, v.amax, p.W, 1);
        lds = std::max(lds, tile_lds(p.AE, p.W, 1));
        dj[i].sino = j.sino;
        dj[i].img = j.img;
        dj[i].lut_off = h->lut_off[i];
        dj[i].in_f16 = j.dtype == RISA_F16 ? 1 : 0;
        dj[i].p = p;
        const float c = p.center;
        for (int t = 0; t < p.tilesX * tilesY; t++) {
            const int x0 = (t % p.tilesX) * v.tx, y0 = (t / p.tilesX) * v.ty;
            // pixels of the tile inside the image (and the circle when masked)
            long px = 0;
            for (int y = y0; y < std::min(j.N, y0 + v.ty); y += 4)
                for (int x = x0; x < std::min(j.N, x0 + v.tx); x += 4) {
                    const float dX = (float)x - c, dY = (float)y - c;
                    if (!p.mask || (double)(dX * dX + dY * dY) <= (double)j.N * j.N * 0.25) px++;
                }
            order.push_back({px * (long)j.P, make_int2((int)i, t)});
        }
    }
    std::stable_sort(order.begin(), order.end(), [](const auto& a, const auto& b) { return a.first > b.first; });
    std::vector<int2> tl(order.size());
    for (size_t i = 0; i < order.size(); i++) tl[i] = order[i].second;
    if (lds > kMaxLds) fail(RISA_ERR_UNSUPPORTED, "backprojection tiles need %zu B of LDS", lds);
    h->ntiles = (int)tl.size();
    h->lds = lds;
    h->djobs.resize(dj.size());
    h->djobs.upload(dj);
    h->tiles.resize(tl.size());
    h->tiles.upload(tl);
    int cus = 0, per_cu = 0;
    RISA_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, h->device));
    RISA_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(v.fn),
                                                                 v.tx * v.ty / v.ppt, h->lds));
    h->grid = std::max(1, std::min(h->ntiles, cus * std::max(1, per_cu)));
}

extern "C" int risa_hip_bp_batched_create(const risa_bp_job* jobs, int njobs, int device, risa_bp_batched_t* out)
{
    return guarded("risa_hip_bp_batched_create", [&] {
        if (!jobs || njobs <= 0 || !out) fail(RISA_ERR_ARG, "bad argument");
        DeviceGuard dg(device);
        auto h = new risa_bp_batched_s();
        try {
            h->device = device;
            h->jobs.assign(jobs, jobs + njobs);
            std::vector<float> cs, sn;
            for (int i = 0; i < njobs; i++) {
                const risa_bp_job& j = jobs[i];
                if (j.N <= 0 || j.P <= 0 || j.D <= 0 || !j.sino || !j.img) fail(RISA_ERR_ARG, "job %d is invalid", i);
                if (j.dtype != RISA_F32 && j.dtype != RISA_F16) fail(RISA_ERR_ARG, "job %d: unknown dtype", i);
                if (j.dtype == RISA_F16 && !(j.in_scale > 0)) fail(RISA_ERR_ARG, "job %d: in_scale must be > 0", i);
                risa_geom g{};
                g.numberOfParallelProjections = j.P;
                g.numberOfParallelDetectors = j.D;
                g.numberOfPixels = j.N;
                g.rotationOffset = j.rotationOffset;
                const BpLut l = bp_lut(g);
                h->lut_off.push_back((int)cs.size());
                cs.insert(cs.end(), l.cosT.begin(), l.cosT.end());
                sn.insert(sn.end(), l.sinT.begin(), l.sinT.end());
            }
            h->cosT.resize(cs.size());
            h->cosT.upload(cs);
            h->sinT.resize(sn.size());
            h->sinT.upload(sn);
            h->counter.resize(1);
            // the first tile shape that holds every job's windows
            for (;; h->variant++) {
                try {
                    batched_layout(h);
                    break;
                } catch (const Error& e) {
                    if (e.code != RISA_ERR_UNSUPPORTED || h->variant + 1 >= kNumPersistent) throw;
                }
            }
        } catch (...) {
            delete h;
            throw;
        }
        *out = h;
    });
}

extern "C" int risa_hip_bp_batched_set_buffers(risa_bp_batched_t h, const risa_bp_job* jobs, int njobs)
{
    return guarded("risa_hip_bp_batched_set_buffers", [&] {
        if (!h || !jobs || njobs != (int)h->jobs.size()) fail(RISA_ERR_ARG, "job count mismatch");
        for (int i = 0; i < njobs; i++) {
            const risa_bp_job& a = h->jobs[i];
            const risa_bp_job& b = jobs[i];
            if (a.N != b.N || a.P != b.P || a.D != b.D || a.dtype != b.dtype) fail(RISA_ERR_ARG, "job %d geometry changed", i);
            h->jobs[i].sino = b.sino;
            h->jobs[i].img = b.img;
        }
        DeviceGuard dg(h->device);
        batched_layout(h);
    });
}

static void launch_persistent(risa_bp_batched_t h, hipStream_t s)
{
    const PersistentVariant& v = kPersistent[h->variant];
    hipLaunchKernelGGL(reset_counter_kernel, dim3(1), dim3(1), 0, s, h->counter.ptr);
    check_launch("reset_counter_kernel");
    hipLaunchKernelGGL(v.fn, dim3(h->grid), dim3(v.tx * v.ty / v.ppt), h->lds, s, h->djobs.ptr, h->tiles.ptr,
                       h->ntiles, h->cosT.ptr, h->sinT.ptr, h->counter.ptr);
    check_launch("bp_persistent_kernel");
}

extern "C" int risa_hip_bp_batched_run(risa_bp_batched_t h, void* stream)
{
    return guarded("risa_hip_bp_batched_run", [&] {
        if (!h) fail(RISA_ERR_ARG, "null handle");
        launch_persistent(h, as_stream(stream));
    });
}

extern "C" int risa_hip_bp_batched_set_variant(risa_bp_batched_t h, int variant)
{
    return guarded("risa_hip_bp_batched_set_variant", [&] {
        if (!h || variant < 0 || variant >= kNumPersistent) fail(RISA_ERR_ARG, "variant out of range");
        DeviceGuard dg(h->device);
        const int before = h->variant;
        h->variant = variant;
        try {
            batched_layout(h);
        } catch (...) {
            h->variant = before;   // the layout is still that variant's
            throw;
        }
    });
}

// Autotuner over the persistent tile shapes: times each on the real jobs.
extern "C" int risa_hip_bp_batched_autotune(risa_bp_batched_t h, void* stream)
{
    return guarded("risa_hip_bp_batched_autotune", [&] {
        if (!h) fail(RISA_ERR_ARG, "null handle");
        DeviceGuard dg(h->device);
        hipStream_t s = as_stream(stream);
        hipEvent_t e0, e1;
        RISA_HIP_CHECK(hipEventCreate(&e0));
        RISA_HIP_CHECK(hipEventCreate(&e1));
        float best = 1e30f;
        int bestv = 0;
        for (int v = 0; v < kNumPersistent; v++) {
            h->variant = v;
            try {
                batched_layout(h);
            } catch (const Error&) {
                continue;
            }
            launch_persistent(h, s);
            RISA_HIP_CHECK(hipEventRecord(e0, s));
            for (int it = 0; it < 3; it++) launch_persistent(h, s);
            RISA_HIP_CHECK(hipEventRecord(e1, s));
            RISA_HIP_CHECK(hipEventSynchronize(e1));
            float ms = 0;
            RISA_HIP_CHECK(hipEventElapsedTime(&ms, e0, e1));
            if (ms < best) { best = ms; bestv = v; }
        }
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        h->variant = bestv;
        batched_layout(h);
    });
}

extern "C" int risa_hip_bp_batched_destroy(risa_bp_batched_t h)
{
    return guarded("risa_hip_bp_batched_destroy", [&] {
        if (h) drain_device(h->device);
        delete h;
    });
}
