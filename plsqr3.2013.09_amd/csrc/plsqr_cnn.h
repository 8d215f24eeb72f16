// Device kernels of the warm-start network (included once, by plsqr_cnn.hip).
//
// A 3-D convolutional network maps the back-projection A^T b on the voxel
// grid to a starting point x0 for LSQR.  Every activation has C = 32 channels
// stored channels-last as bf16, element (g, c) at g*C + c with g = b*V + v the
// (sample, voxel) index; the network's one input and one output channel are
// channel 0 of a 32-channel tensor whose other channels are zero (input) or
// ignored (output), so that every layer is the same 32 -> 32 convolution.
// Those two tensors, and the gradient of the output, are stored as that one
// channel (FP32 [g]); the kernels supply the zeros.
//
// A 3x3x3 convolution with zero padding is an implicit GEMM: M = 32 output
// channels, N = voxels, K = 27 taps x 32 input channels, in steps of one
// v_mfma_f32_32x32x16_bf16 (bf16 operands, FP32 accumulation):
//   A (32 x 16): lane l holds row l%32, k = 8*(l/32) .. +7
//   B (16 x 32): lane l holds column l%32, k = 8*(l/32) .. +7
//   D (32 x 32): lane l, register r holds row 8*(r/4) + 4*(l/32) + r%4,
//                column l%32
// Weights are bf16 in [tap][out channel][in channel] order so that a lane's
// eight k values are contiguous.  Tap t = (dz+1)*9 + (dy+1)*3 + (dx+1) reads
// the neighbour at (x+dx, y+dy, z+dz); tap 26-t is its mirror.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace plsqr {
namespace cnn {

constexpr int C = 32;
constexpr int TAPS = 27;

typedef short short4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t uint4_t __attribute__((ext_vector_type(4)));
typedef uint32_t uint2_t __attribute__((ext_vector_type(2)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

// float -> bf16 bits, round to nearest even (v_cvt_pk_bf16_f32)
__device__ __forceinline__ uint16_t f2bf(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }

__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// two floats as packed bf16 bits, the first in the low half
__device__ __forceinline__ uint32_t pack_bf(float lo, float hi) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, bf16x2{(__bf16)lo, (__bf16)hi});
}

// ---------------------------------------------------------------------------
// out[g][n] = f(bias[n] + sum_t sum_k in[g + off(t)][k] * w[t][n][k]) for the
// (sample, voxel) rows g of `samples` grids; neighbours outside the grid read
// as zero.  f: ReLU when relu != 0; then, when mask is given, out = 0 where
// mask[g][n] <= 0 (the ReLU derivative of the layer below, for the data
// gradient; with OUT = CONV_BF16 only).
//   IN   CONV_BF16 bf16 [g][32]; CONV_F32 FP32 [g][32], rounded to bf16 here;
//        CONV_ONE FP32 [g], channel 0 of an input whose other channels are
//        zero (their K steps, which would add zeros, are left out)
//   WF32 the weights are FP32 (rounded here) instead of bf16
//   OUT  CONV_BF16 bf16 [g][32], CONV_F32 FP32 [g][32] or CONV_ONE FP32 [g]
//        (channel 0)
//
// A workgroup owns bricks of 8 x 8 x 8 voxels: the 10 x 10 x 10 neighbourhood
// and all weights lie in LDS, so each input row is read from memory about
// twice instead of 27 times and the 27 taps are LDS reads at constant offsets
// from one address per lane.  Wavefront w computes plane w of the brick as two
// 32-voxel columns (8 x 4) that share each weight fragment.  With only the LDS
// reads and matrix steps left the kernel takes 59 us of the 87 below (1.13
// PFLOP/s; a large matrix product reaches 1.36).  A voxel takes 80 bytes of LDS
// for its 64 and a line of voxels 896, so that the 16-byte reads of 16 lanes (8
// in x, 2 in y) fall on different banks (with lines of 800 bytes half of the LDS cycles were conflicts: 118 us).  One
// workgroup per CU stays for all of its bricks (weights are staged
// once); the next brick's rows are loaded into registers while this one is
// summed.  Workgroup b takes bricks of the b % 8-th of eight contiguous ranges,
// so neighbouring bricks share their halo in one XCD's L2.
// 48^3, FP32 in and out: 16.2 us, 65 before (fragments loaded from
// memory per tap: 56 us, and two passes that made bf16 copies); 67^3 x 4
// samples, bf16: 87 us per layer, 478 before.
// ---------------------------------------------------------------------------
enum { CONV_BF16 = 0, CONV_F32 = 1, CONV_ONE = 2 };
constexpr int CB = 8;                    // brick edge
constexpr int CH = CB + 2;               // with its halo
constexpr int CONV_THREADS = 64 * CB;    // one wavefront per plane

template <int IN, bool WF32, int OUT>
__global__ __launch_bounds__(CONV_THREADS, 2) void kc_conv(int nx, int ny, int nz, int samples, const void *__restrict__ in,
                                                           const void *__restrict__ w, const float *__restrict__ bias,
                                                           const uint16_t *__restrict__ mask, int relu,
                                                           void *__restrict__ out, int aligned) {
    constexpr int KS = IN == CONV_ONE ? 1 : 2;       // K steps per tap
    constexpr int VS = IN == CONV_ONE ? 3 : 5;       // 16-byte units per voxel in LDS (2 or 4 of data)
    constexpr int CPV = IN == CONV_ONE ? 1 : 4;      // units loaded per voxel
    constexpr int NV = CH * CH * CH;
    // units per line and plane of the neighbourhood: a line is 8 (mod 16) units
    // long, so the 16 lanes of a read cycle (8 in x, 2 in y) take 16 bank groups
    constexpr int LP = IN == CONV_ONE ? 40 : 56, PP = CH * LP;
    static_assert(LP >= CH * VS && LP % 16 == 8, "lines do not overlap and fall on different banks");
    constexpr int PER = (NV * CPV + CONV_THREADS - 1) / CONV_THREADS;
    __shared__ uint4_t wl[TAPS * KS * 64];
    __shared__ uint4_t xl[CH * PP];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int tx = (nx + CB - 1) / CB, ty = (ny + CB - 1) / CB, tz = (nz + CB - 1) / CB;
    const int per_sample = tx * ty * tz, tiles = per_sample * samples;
    // this workgroup's bricks: first, first + step, ... below last
    const int queues = gridDim.x % 8 == 0 ? 8 : 1;
    const int q = blockIdx.x % queues, step = gridDim.x / queues;
    const int first = (int)((long long)tiles * q / queues) + blockIdx.x / queues;
    const int last = (int)((long long)tiles * (q + 1) / queues);
    if (first >= last) return;

    // weight fragments, lane-linear: unit (t * KS + s) * 64 + l holds w[t][l%32][16 s + 8 (l/32) .. +7]
    {
        constexpr int NU = TAPS * KS * 64, WPER = (NU + CONV_THREADS - 1) / CONV_THREADS;
        uint4_t u[WPER][WF32 ? 2 : 1];
        const bool wide = ((uintptr_t)w & 15) == 0;
#pragma unroll
        for (int j = 0; j < WPER; ++j) {
            const int i = min(tid + j * CONV_THREADS, NU - 1);
            const int l = i & 63, s = (i >> 6) % KS, t = (i >> 6) / KS;
            const int src = (t * C + (l & 31)) * C + 16 * s + 8 * (l >> 5);
            if constexpr (!WF32) {
                u[j][0] = *(const uint4_t *)((const uint16_t *)w + src);
            } else if (wide) {
                u[j][0] = ((const uint4_t *)((const float *)w + src))[0];
                u[j][1] = ((const uint4_t *)((const float *)w + src))[1];
            } else {
#pragma unroll
                for (int k = 0; k < 8; ++k) u[j][k / 4][k % 4] = ((const uint32_t *)w)[src + k];
            }
        }
#pragma unroll
        for (int j = 0; j < WPER; ++j) {
            const int i = tid + j * CONV_THREADS;
            if constexpr (WF32) {
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    u[j][0][k] = pack_bf(__uint_as_float(u[j][k / 2][2 * (k % 2)]), __uint_as_float(u[j][k / 2][2 * (k % 2) + 1]));
            }
            if (i < NU) wl[i] = u[j][0];
        }
    }
    if constexpr (IN == CONV_ONE)  // channels 8..15 are zero
        for (int p = tid; p < NV; p += CONV_THREADS)
            xl[p / (CH * CH) * PP + p / CH % CH * LP + p % CH * VS + 1] = uint4_t{0, 0, 0, 0};

    // the neighbourhood of a brick: loads into registers, then LDS
    constexpr int RU = IN == CONV_F32 ? 2 : 1;
    uint4_t reg[PER][RU];
    // per unit, kept for all bricks: its voxel in the neighbourhood (bytes x, y,
    // z) and its offset from the neighbourhood's first row, in units
    int at[PER];
    uint32_t off[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int i = tid + j * CONV_THREADS;
        const int p = min(i / CPV, NV - 1), c = i % CPV;
        const int px = p % CH, py = p / CH % CH, pz = p / (CH * CH);
        at[j] = px | py << 8 | pz << 16;
        off[j] = (uint32_t)((pz * ny + py) * nx + px) * CPV + c;
    }
    const uint32_t centre = (uint32_t)((ny + 1) * nx + 1) * CPV;  // a row of the brick itself
    auto load = [&](int tile) {
        const int sample = tile / per_sample, r = tile % per_sample;
        const int x0 = (r % tx) * CB - 1, y0 = (r / tx % ty) * CB - 1, z0 = (r / (tx * ty)) * CB - 1;
        const long long first_row = (((long long)sample * nz + z0) * ny + y0) * nx + x0;
        constexpr int UB = IN == CONV_BF16 ? 16 : IN == CONV_F32 ? 32 : 4;  // bytes of a unit in memory
        const uintptr_t from = (uintptr_t)in + first_row * (UB * CPV);
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const bool ok = (unsigned)(x0 + (at[j] & 255)) < (unsigned)nx && (unsigned)(y0 + (at[j] >> 8 & 255)) < (unsigned)ny &&
                            (unsigned)(z0 + (at[j] >> 16)) < (unsigned)nz;
            // outside: load a row of the brick and drop it (a predicated load would wait for itself)
            const uintptr_t src = from + (uintptr_t)(ok ? off[j] : centre) * UB;
            if constexpr (IN == CONV_BF16) {
                reg[j][0] = *(const uint4_t *)src;
                if (!ok) reg[j][0] = uint4_t{0, 0, 0, 0};
            } else if constexpr (IN == CONV_F32) {
                if (aligned) {
                    reg[j][0] = ((const uint4_t *)src)[0];
                    reg[j][1] = ((const uint4_t *)src)[1];
                } else {
#pragma unroll
                    for (int k = 0; k < 8; ++k) reg[j][k / 4][k % 4] = ((const uint32_t *)src)[k];
                }
                if (!ok) reg[j][0] = reg[j][1] = uint4_t{0, 0, 0, 0};
            } else {
                const uint32_t f = *(const uint32_t *)src;
                reg[j][0][0] = ok ? f : 0u;
            }
        }
    };
    auto store = [&]() {
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int i = tid + j * CONV_THREADS;
            if (i >= NV * CPV) break;
            const int to = (at[j] >> 16) * PP + (at[j] >> 8 & 255) * LP + (at[j] & 255) * VS + i % CPV;
            uint4_t u = reg[j][0];
            if constexpr (IN == CONV_F32) {
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    u[k] = pack_bf(__uint_as_float(reg[j][k / 2][2 * (k % 2)]), __uint_as_float(reg[j][k / 2][2 * (k % 2) + 1]));
            } else if constexpr (IN == CONV_ONE) {
                u = uint4_t{f2bf(__uint_as_float(reg[j][0][0])), 0, 0, 0};
            }
            xl[to] = u;
        }
    };

    const int i = lane & 31, h = lane >> 5;
    float bn[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) bn[r] = bias ? bias[8 * (r / 4) + 4 * h + r % 4] : 0.f;
    const uint4_t *xa = xl + wave * PP + (i >> 3) * LP + (i & 7) * VS + h;
    load(first);
    for (int tile = first; tile < last; tile += step) {
        store();
        __syncthreads();
        if (tile + step < last) load(tile + step);
        const int sample = tile / per_sample, rr = tile % per_sample;
        const int x = (rr % tx) * CB + (i & 7), yb = (rr / tx % ty) * CB, z = (rr / (tx * ty)) * CB + wave;
        if (z < nz) {  // uniform per wavefront
            floatx16 acc[2];
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[0][r] = acc[1][r] = 0.f;
            const bool two = yb + 4 < ny;
            // the mask rows are loaded before the sums: they would wait for
            // memory after them (67^3 x 4: 119 -> 105 us per layer)
            uint2_t mk[2][4];
            if constexpr (OUT == CONV_BF16) {
                if (mask) {
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const long long g = (((long long)sample * nz + z) * ny + min(yb + 4 * e + (i >> 3), ny - 1)) * nx + min(x, nx - 1);
#pragma unroll
                        for (int b = 0; b < 4; ++b) mk[e][b] = *(const uint2_t *)(mask + g * C + 8 * b + 4 * h);
                    }
                }
            }
            // groups of GS steps (fragments of one tap and K step): one group's
            // fragments are read while the group before it is multiplied
            auto sum = [&](auto halves) {
                constexpr int NH = decltype(halves)::value, GS = 3, NG = TAPS * KS / GS;
                static_assert(NG * GS == TAPS * KS, "whole groups");
                bf16x8 a[2][GS], b[2][GS][NH];
                auto read = [&](int gr) {
#pragma unroll
                    for (int k = 0; k < GS; ++k) {
                        const int f = gr * GS + k, t = f / KS;
                        a[gr & 1][k] = __builtin_bit_cast(bf16x8, wl[f * 64 + lane]);
#pragma unroll
                        for (int e = 0; e < NH; ++e)
                            b[gr & 1][k][e] = __builtin_bit_cast(
                                bf16x8, xa[t / 9 * PP + (t / 3 % 3 + 4 * e) * LP + t % 3 * VS + 2 * (f % KS)]);
                    }
                };
                read(0);
#pragma unroll
                for (int gr = 0; gr < NG; ++gr) {
                    if (gr + 1 < NG) read(gr + 1);
                    __builtin_amdgcn_sched_barrier(0);  // the reads would sink to their uses
#pragma unroll
                    for (int k = 0; k < GS; ++k)
#pragma unroll
                        for (int e = 0; e < NH; ++e)
                            acc[e] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[gr & 1][k], b[gr & 1][k][e], acc[e], 0, 0, 0);
                }
            };
            if (two)
                sum(std::integral_constant<int, 2>{});
            else
                sum(std::integral_constant<int, 1>{});
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int y = yb + 4 * e + (i >> 3);
                if (x >= nx || y >= ny) continue;
                const long long g = (((long long)sample * nz + z) * ny + y) * nx + x;
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    const long long o = g * C + 8 * b + 4 * h;  // channels 8b + 4h .. +3
                    float v[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        v[k] = acc[e][4 * b + k] + bn[4 * b + k];
                        if (relu) v[k] = fmaxf(v[k], 0.f);
                    }
                    if constexpr (OUT == CONV_BF16) {
                        if (mask) {
#pragma unroll
                            for (int k = 0; k < 4; ++k)
                                if (!(bf2f((uint16_t)(mk[e][b][k / 2] >> (16 * (k % 2)))) > 0.f)) v[k] = 0.f;
                        }
                        *(uint2_t *)((uint16_t *)out + o) = uint2_t{pack_bf(v[0], v[1]), pack_bf(v[2], v[3])};
                    } else if constexpr (OUT == CONV_ONE) {
                        if (b == 0 && h == 0) ((float *)out)[g] = v[0];
                    } else {
                        float *d = (float *)out + o;
                        if (aligned) {
                            *(float4 *)d = make_float4(v[0], v[1], v[2], v[3]);
                        } else {
#pragma unroll
                            for (int k = 0; k < 4; ++k) d[k] = v[k];
                        }
                    }
                }
            }
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// The same layer for grids that fill bricks badly: a wavefront takes 32
// consecutive rows whatever their place in the grid, so thin and tiny grids cost
// no matrix steps for voxels that do not exist.  All weights lie in LDS; for one
// dz at a time the wavefront's three runs of 34 consecutive rows (dy -1, 0, 1)
// pass through LDS as bf16, the loads of the next dz in flight while this one is
// multiplied.  What bounds it is staging each row nine times; fragments loaded
// straight from memory, 32 cache lines per load, were bound by the L1 (131072
// voxels, FP32: 69 us, here 23).  A tap without a neighbour multiplies zeros.
// Taps and K steps are added in kc_conv's order, so both give the same bits.
// 120 KB of LDS: one workgroup per CU stays for all of its rows.
// ---------------------------------------------------------------------------
template <int IN, bool WF32, int OUT>
__global__ __launch_bounds__(CONV_THREADS, 2) void kc_conv_rows(int nx, int ny, int nz, unsigned total, const void *__restrict__ in,
                                                                const void *__restrict__ w, const float *__restrict__ bias,
                                                                const uint16_t *__restrict__ mask, int relu,
                                                                void *__restrict__ out, int aligned) {
    constexpr int KS = IN == CONV_ONE ? 1 : 2;
    constexpr int RUN = 34;                                            // rows of a run
    constexpr int PIECES = IN == CONV_F32 ? 8 : IN == CONV_BF16 ? 4 : 1;  // loads per row: four floats, eight bf16 or one float
    constexpr int PER = (RUN * PIECES + 63) / 64;
    constexpr int VS = IN == CONV_ONE ? 1 : 5;                         // 16-byte units per row in LDS (4 of data)
    __shared__ uint4_t wl[TAPS * KS * 64];
    __shared__ uint4_t xs[CB][3][RUN * VS];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i = lane & 31, h = lane >> 5;
    // weight fragments as in kc_conv
    const bool wide = ((uintptr_t)w & 15) == 0;
#pragma unroll
    for (int j = 0; j < (TAPS * KS * 64 + CONV_THREADS - 1) / CONV_THREADS; ++j) {
        const int f = threadIdx.x + j * CONV_THREADS;
        if (f >= TAPS * KS * 64) break;
        const int src = ((f >> 6) / KS * C + (f & 31)) * C + 16 * ((f >> 6) % KS) + 8 * (f >> 5 & 1);
        if constexpr (!WF32) {
            wl[f] = *(const uint4_t *)((const uint16_t *)w + src);
        } else {
            const float *p = (const float *)w + src;
            float4 a, b;
            if (wide)
                a = ((const float4 *)p)[0], b = ((const float4 *)p)[1];
            else
                a = make_float4(p[0], p[1], p[2], p[3]), b = make_float4(p[4], p[5], p[6], p[7]);
            wl[f] = uint4_t{pack_bf(a.x, a.y), pack_bf(a.z, a.w), pack_bf(b.x, b.y), pack_bf(b.z, b.w)};
        }
    }
    float bn[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) bn[r] = bias ? bias[8 * (r / 4) + 4 * h + r % 4] : 0.f;
    __syncthreads();
    const unsigned groups = (total + 31) / 32;
    for (unsigned gr = blockIdx.x * CB + wave; gr < groups; gr += gridDim.x * CB) {
        const unsigned g = min(gr * 32 + i, total - 1);  // past the end: the last row again, not stored
        const unsigned line = g / (unsigned)nx, plane = line / (unsigned)ny;
        const int x = (int)(g - line * nx), y = (int)(line - plane * ny), z = (int)(plane % (unsigned)nz);
        uint2_t mk[4];
        if constexpr (OUT == CONV_BF16) {
            if (mask) {
#pragma unroll
                for (int b = 0; b < 4; ++b) mk[b] = *(const uint2_t *)(mask + (size_t)g * C + 8 * b + 4 * h);
            }
        }
        uint4_t u[3][PER];
        auto load = [&](int dz) {
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                const long long first = (long long)gr * 32 - 1 + ((long long)dz * ny + q - 1) * nx;
#pragma unroll
                for (int j = 0; j < PER; ++j) {
                    const int p = min(lane + 64 * j, RUN * PIECES - 1);
                    // rows outside the tensor are no row's neighbour
                    const long long r = min(max(first + p / PIECES, 0LL), (long long)total - 1);
                    const long long src = r * PIECES + p % PIECES;
                    if constexpr (IN == CONV_ONE) {
                        u[q][j][0] = ((const uint32_t *)in)[src];
                    } else if (IN == CONV_BF16 || aligned) {
                        u[q][j] = ((const uint4_t *)in)[src];
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e) u[q][j][e] = ((const uint32_t *)in)[src * 4 + e];
                    }
                }
            }
        };
        auto store = [&]() {
#pragma unroll
            for (int q = 0; q < 3; ++q)
#pragma unroll
                for (int j = 0; j < PER; ++j) {
                    const int p = lane + 64 * j, row = p / PIECES, c = p % PIECES;
                    if (p >= RUN * PIECES) break;
                    uint4_t *const to = xs[wave][q] + row * VS;
                    if constexpr (IN == CONV_ONE)
                        to[0] = uint4_t{f2bf(__uint_as_float(u[q][j][0])), 0, 0, 0};
                    else if constexpr (IN == CONV_BF16)
                        to[c] = u[q][j];
                    else
                        ((uint2_t *)to)[c] = uint2_t{pack_bf(__uint_as_float(u[q][j][0]), __uint_as_float(u[q][j][1])),
                                                     pack_bf(__uint_as_float(u[q][j][2]), __uint_as_float(u[q][j][3]))};
                }
        };
        floatx16 acc;
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] = 0.f;
        load(-1);
#pragma unroll 1
        for (int dz = -1; dz <= 1; ++dz) {
            store();
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            if (dz < 1) load(dz + 1);
            const uint4_t *const wt = wl + (dz + 1) * 9 * KS * 64 + lane;
#pragma unroll
            for (int t = 0; t < 9; ++t) {
                const int q = t / 3, dx = t % 3 - 1;
                const bool ok = (unsigned)(z + dz) < (unsigned)nz && (unsigned)(y + q - 1) < (unsigned)ny && (unsigned)(x + dx) < (unsigned)nx;
#pragma unroll
                for (int s = 0; s < KS; ++s) {
                    uint4_t b = xs[wave][q][(i + t % 3) * VS + (IN == CONV_ONE ? 0 : 2 * s + h)];
                    if (!ok || (IN == CONV_ONE && h == 1)) b = uint4_t{0, 0, 0, 0};
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, wt[(t * KS + s) * 64]),
                                                                  __builtin_bit_cast(bf16x8, b), acc, 0, 0, 0);
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
        if (gr * 32 + i >= total) continue;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const size_t o = (size_t)g * C + 8 * b + 4 * h;  // channels 8b + 4h .. +3
            float v[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                v[k] = acc[4 * b + k] + bn[4 * b + k];
                if (relu) v[k] = fmaxf(v[k], 0.f);
            }
            if constexpr (OUT == CONV_BF16) {
                if (mask) {
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        if (!(bf2f((uint16_t)(mk[b][k / 2] >> (16 * (k % 2)))) > 0.f)) v[k] = 0.f;
                }
                *(uint2_t *)((uint16_t *)out + o) = uint2_t{pack_bf(v[0], v[1]), pack_bf(v[2], v[3])};
            } else if constexpr (OUT == CONV_ONE) {
                if (b == 0 && h == 0) ((float *)out)[g] = v[0];
            } else {
                float *d = (float *)out + o;
                if (aligned) {
                    *(float4 *)d = make_float4(v[0], v[1], v[2], v[3]);
                } else {
#pragma unroll
                    for (int k = 0; k < 4; ++k) d[k] = v[k];
                }
            }
        }
    }
}

// s + this thread's rows q, q + 8, .. of the first `live` rows of staged dout
// (a multiple of 64 rows is readable), thread (q, n) = (tid / 32, tid % 32)
__device__ __forceinline__ float bias_rows(float s, const uint16_t *rows, int live) {
    for (int r = threadIdx.x / C; r < live; r += 64) {
        float v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = bf2f(rows[(r + 8 * k) * C + threadIdx.x % C]);
#pragma unroll
        for (int k = 0; k < 8; ++k)
            if (r + 8 * k < live) s += v[k];
    }
    return s;
}

// A chunk's bias gradient: thread (q, n) = (tid / 32, tid % 32) holds the sum s
// of rows q, q + 8, ..; the eight are added in order.  red: 256 floats of LDS.
__device__ __forceinline__ void bias_partial(float s, float *red, float *__restrict__ part) {
    red[threadIdx.x] = s;
    __syncthreads();
    if (threadIdx.x < C) {
        float r = 0.f;
        for (int k = 0; k < 8; ++k) r += red[k * C + threadIdx.x];
        part[threadIdx.x] = r;
    }
}

// ---------------------------------------------------------------------------
// Weight gradient: part[t * nch + chunk][n][k] = sum over the chunk's rows g of
// dout[g][n] * in[g + off(t)][k] (neighbours outside the grid are zero), and the
// bias gradient's partials bpart[chunk][n].  DONE: dout is one channel, FP32
// [g].  A wavefront w adds rows 8w .. 8w+7 of every 32 (the matrix reduction
// dimension is rows, two such steps per 32x32x16), and the four wavefronts'
// sums are added in order.
//
// TG taps per workgroup: 9 (one dz) or 3 (one dz and dy); one dout fragment
// serves them all.  Sub-blocks of 256 rows of dout and the contiguous rows of
// `in` that their taps read are staged in LDS (a thread's loads for the next
// sub-block are in flight while this one is multiplied), and
// ds_read_b64_tr_b16 gives each lane four rows of its channel, which lie
// across the channels in memory.  A tap is one offset from the row; near[r]
// says which of a row's neighbours exist, and a tap without one reads a row of
// zeros.  (Staging zero-padded lines instead needs no test, but finding each
// staged row's place took 112 of 200 vector instructions per 9 matrix steps,
// 182 us; loading both operands two bytes at a time from memory, tap by tap,
// took 1783 us.)
// 67^3 x 4 samples: 132 us per layer, 140 with a one-channel dout.
//
// Workgroup b works in the b % 8-th of eight contiguous ranges of chunks, so
// the tap groups of a chunk and its neighbours share an XCD's L2.  The host
// takes nine taps when lines are short enough for LDS and there are chunks
// enough to fill the chip.
// ---------------------------------------------------------------------------
constexpr int WGRAD_R = 256;       // rows of dout per sub-block
constexpr int WGRAD_XROWS = 640;   // staged rows of `in`: WGRAD_R + 2 (nx + 1) with nine taps
constexpr int WGRAD_NX9 = (WGRAD_XROWS - WGRAD_R - 2) / 2;

template <int TG, bool DONE>
__global__ __launch_bounds__(256, 2) void kc_wgrad(int nx, int ny, int nz, long long total, int chunk_len,
                                                   const uint16_t *__restrict__ in, const void *__restrict__ dout,
                                                   float *__restrict__ part, float *__restrict__ bpart) {
    static_assert(TG == 3 || TG == 9, "the taps of one (dz, dy) or of one dz");
    constexpr int GROUPS = TAPS / TG, R = WGRAD_R;
    constexpr int XROWS = TG == 9 ? WGRAD_XROWS : R + 64, PA = R * 4 / 256, PX = XROWS * 4 / 256;
    // bits of near[]: x-1, x+1, y-1, y+1 exist; the row is in the chunk and z+dz in the grid
    __shared__ uint4_t da[R * 4];
    __shared__ uint4_t xa[(XROWS + 1) * 4];  // the last row: zeros
    __shared__ uint8_t near[R];
    static_assert(sizeof(da) >= 4 * C * C * sizeof(float), "the wavefronts' sums pass through da");
    const int nch = (int)((total + chunk_len - 1) / chunk_len), jobs = nch * GROUPS;
    const int q = blockIdx.x % 8, job = (int)((long long)jobs * q / 8) + blockIdx.x / 8;
    if (job >= (int)((long long)jobs * (q + 1) / 8)) return;
    const int chunk = job / GROUPS, group = job % GROUPS;
    const int dz = (TG == 9 ? group : group / 3) - 1, dline = TG == 9 ? 0 : group % 3 - 1;
    const int halo = (TG == 9 ? nx : 0) + 1, xunits = (R + 2 * halo) * 4;
    const long long shift = ((long long)dz * ny + dline) * nx;  // row of the group's middle tap
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int s16 = lane & 15, h = lane >> 5, i = lane & 31;
    const int lrow = wave * 8 + 32 * h + (s16 >> 2);              // this lane's row of a step's first four
    const int lbyte = ((lane >> 4) & 1) * 32 + (s16 & 3) * 8;     // its channels in the row
    typedef __attribute__((address_space(3))) short4_t lds_short4;
    typedef __attribute__((address_space(3))) char lds_char;
    lds_char *const dl = (lds_char *)da + lbyte, *const xb = (lds_char *)xa + lbyte;
    lds_char *const zeros = xb + XROWS * (C * 2);
    auto transposed = [](lds_char *p) { return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4 *)p); };
    const long long c0 = (long long)chunk * chunk_len, c1 = min(c0 + chunk_len, total);
    uint4_t ua[PA], ux[PX];
    auto load = [&](long long s) {
        const int live = (int)min((long long)R, c1 - s);
#pragma unroll
        for (int k = 0; k < PA; ++k) {
            const int unit = min(tid + k * 256, live * 4 - 1);
            if constexpr (DONE)
                ua[k] = uint4_t{unit % 4 == 0 ? f2bf(((const float *)dout)[s + unit / 4]) : 0u, 0, 0, 0};
            else
                ua[k] = ((const uint4_t *)dout + s * 4)[unit];
            if (tid + k * 256 >= live * 4) ua[k] = uint4_t{0, 0, 0, 0};
        }
        // rows s + shift - halo .., clamped to the tensor (rows outside it are never
        // used; a run wholly outside is moved to its end)
        const long long r0 = min(max(s + shift - halo, 1LL - XROWS), total - 1);
        const int lo = (int)max(-r0, 0LL) * 4, hi = (int)min(total - r0, (long long)XROWS) * 4 - 1;
        const uint4_t *from = (const uint4_t *)in + r0 * 4;
#pragma unroll
        for (int k = 0; k < PX; ++k)
            if (k * 256 < xunits) ux[k] = from[min(max(tid + k * 256, lo), hi)];
    };
    floatx16 acc[TG];
#pragma unroll
    for (int t = 0; t < TG; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[t][r] = 0.f;
    float bsum = 0.f;
    // this thread's row: its voxel, advanced by R rows per sub-block
    const long long l0 = (c0 + tid) / nx, p0 = l0 / ny;
    int vx = (int)(c0 + tid - l0 * nx), vy = (int)(l0 - p0 * ny), vz = (int)(p0 % nz);
    const int sx = R % nx, sy = R / nx % ny, sz = R / nx / ny % nz;
    if (tid < 4) xa[XROWS * 4 + tid] = uint4_t{0, 0, 0, 0};
    load(c0);
#pragma unroll 1
    for (long long s = c0; s < c1; s += R) {
        const int live = (int)min((long long)R, c1 - s);
#pragma unroll
        for (int k = 0; k < PA; ++k) da[tid + k * 256] = ua[k];
#pragma unroll
        for (int k = 0; k < PX; ++k)
            if (k * 256 < xunits) xa[tid + k * 256] = ux[k];
        near[tid] = (uint8_t)((vx > 0 ? 1 : 0) | (vx < nx - 1 ? 2 : 0) | (vy > 0 ? 4 : 0) | (vy < ny - 1 ? 8 : 0) |
                              (tid < live && (unsigned)(vz + dz) < (unsigned)nz ? 16 : 0));
        vx += sx;
        vy += sy;
        vz += sz;
        if (vx >= nx) {
            vx -= nx;
            ++vy;
        }
        if (vy >= ny) {
            vy -= ny;
            ++vz;
        }
        if (vz >= nz) vz -= nz;
        __syncthreads();
        if (s + R < c1) load(s + R);
        if (group == GROUPS / 2) bsum = bias_rows(bsum, (const uint16_t *)da, live);
#pragma unroll 1
        for (int r0 = 0; r0 < live; r0 += 64) {
            typedef short short8_t __attribute__((ext_vector_type(8)));
            short4_t af[2];
            lds_char *x[2];  // first staged row of the tap group's first line, (dy, -1)
            int has[2];
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                const int r = r0 + lrow + 4 * p;
                af[p] = transposed(dl + r * (C * 2));
                has[p] = near[r];
                x[p] = xb + r * (C * 2);
            }
            const bf16x8 a = __builtin_bit_cast(bf16x8, __builtin_shufflevector(af[0], af[1], 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
            for (int dy = 0; dy < TG / 3; ++dy) {
                const int ly = TG == 9 ? dy - 1 : dline, need = 16 | (ly < 0 ? 4 : ly > 0 ? 8 : 0);
                short4_t bf[3][2];
#pragma unroll
                for (int p = 0; p < 2; ++p) {
                    // a tap whose neighbour does not exist reads the row of zeros
                    const bool in_y = (has[p] & need) == need;
                    bf[0][p] = transposed(in_y && (has[p] & 1) ? x[p] : zeros);
                    bf[1][p] = transposed((in_y ? x[p] : zeros - C * 2) + C * 2);
                    bf[2][p] = transposed((in_y && (has[p] & 2) ? x[p] : zeros - 2 * C * 2) + 2 * C * 2);
                    x[p] += nx * (C * 2);
                }
#pragma unroll
                for (int dx = 0; dx < 3; ++dx) {
                    const short8_t b = __builtin_shufflevector(bf[dx][0], bf[dx][1], 0, 1, 2, 3, 4, 5, 6, 7);
                    acc[dy * 3 + dx] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, __builtin_bit_cast(bf16x8, b),
                                                                               acc[dy * 3 + dx], 0, 0, 0);
                }
            }
        }
        __syncthreads();
    }
    float *red = (float *)da;
    if (group == GROUPS / 2) {
        bias_partial(bsum, red, bpart + (size_t)chunk * C);
        __syncthreads();
    }
    // the four wavefronts' sums in order
#pragma unroll
    for (int t = 0; t < TG; ++t) {
#pragma unroll
        for (int r = 0; r < 16; ++r) red[wave * C * C + (8 * (r / 4) + 4 * h + r % 4) * C + i] = acc[t][r];
        __syncthreads();
        float *dst = part + ((size_t)(group * TG + t) * nch + chunk) * (C * C);
        for (int e = tid; e < C * C; e += 256)
            dst[e] = ((red[e] + red[C * C + e]) + red[2 * C * C + e]) + red[3 * C * C + e];
        __syncthreads();
    }
}

// p[0] + p[stride] + .. (count terms, in order), FLIGHT loads in flight: the
// last repeated past the end and not added
template <int FLIGHT>
__device__ __forceinline__ float ordered_sum(const float *__restrict__ p, int count, size_t stride) {
    float s = 0.f;
    for (int c = 0; c < count; c += FLIGHT) {
        float v[FLIGHT];
#pragma unroll
        for (int k = 0; k < FLIGHT; ++k) v[k] = p[(size_t)min(c + k, count - 1) * stride];
#pragma unroll
        for (int k = 0; k < FLIGHT; ++k)
            if (c + k < count) s += v[k];
    }
    return s;
}

// Sums over chunks in order.  Weights: grad[t][n][k] of part[t][chunk][n][k],
// or with FIRST the one channel's grad[t][n][0] of part[chunk][n][t].  Bias
// (the last workgroup): bgrad[n] of bpart[chunk][n].  Each sum is serial and
// there are few of them (27 x 1024), so the loads in flight set the time: 48
// per thread, in one-wavefront workgroups that reach all CUs (67^3 x 4: 294
// chunks, 16.3 -> 9.4 us; 16 per thread in 256-thread workgroups before,
// 71 us with one).
constexpr int GRAD_RED = 64;  // threads per workgroup

template <bool FIRST>
__global__ __launch_bounds__(GRAD_RED) void kc_grad_reduce(int nchunk, const float *__restrict__ part,
                                                           const float *__restrict__ bpart, float *__restrict__ grad,
                                                           float *__restrict__ bgrad) {
    constexpr int F = 48;
    const int idx = blockIdx.x * GRAD_RED + threadIdx.x;
    if (blockIdx.x == gridDim.x - 1) {
        if (threadIdx.x < C) bgrad[threadIdx.x] = ordered_sum<F>(bpart + threadIdx.x, nchunk, C);
    } else if constexpr (FIRST) {
        const int n = idx / C, t = idx % C;
        if (n < C && t < TAPS) grad[(t * C + n) * C] = ordered_sum<F>(part + idx, nchunk, C * C);
    } else {
        const int t = idx / (C * C), e = idx % (C * C);
        if (t < TAPS) grad[idx] = ordered_sum<F>(part + (size_t)t * nchunk * (C * C) + e, nchunk, C * C);
    }
}

// ---------------------------------------------------------------------------
// Weight gradient of the first layer, whose input has one channel (FP32 [g]):
// the 27 taps of that channel are the columns of one 32 x 32 product (the
// other 31 channels' gradients are zero), so a chunk needs one matrix step
// per 16 rows instead of 27 and no 32-channel copy of the input.  Rows are
// added in kc_wgrad's order; part[chunk][n][t], and the bias partials.
// Per sub-block of 256 rows: dout, read transposed; for each (dz, dy) the 258
// inputs its three taps read; and one byte per row that says which neighbours
// exist.  Lane (tap t) gathers its eight rows' inputs from LDS; the next
// sub-block's loads are in flight meanwhile.  67^3 x 4 samples: 46 us
// (kc_wgrad on a 32-channel copy: 132, and 41 for the copy).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void kc_wgrad_first(int nx, int ny, int nz, long long total, int chunk_len,
                                                      const float *__restrict__ x, const uint16_t *__restrict__ dout,
                                                      float *__restrict__ part, float *__restrict__ bpart) {
    constexpr int R = 256, WIN = R + 4;
    __shared__ uint4_t da[R * 4];
    __shared__ float win[9][WIN];
    __shared__ __align__(8) uint8_t near[R];
    static_assert(sizeof(da) >= 4 * C * C * sizeof(float), "the wavefronts' sums pass through da");
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int i = lane & 31, h = lane >> 5, s16 = lane & 15;
    const int dz = i / 9 - 1, dy = i / 3 % 3 - 1, dx = i % 3 - 1;  // columns 27..31: no tap
    // bits of near[]: the row is in the chunk; its neighbours at x-1, x+1, y-1, y+1, z-1, z+1 exist
    const unsigned need = (i < TAPS ? 1u : 128u) | (dx < 0 ? 2u : dx > 0 ? 4u : 0u) | (dy < 0 ? 8u : dy > 0 ? 16u : 0u) |
                          (dz < 0 ? 32u : dz > 0 ? 64u : 0u);
    const float *xw = &win[i < TAPS ? i / 3 : 0][1 + dx];
    typedef __attribute__((address_space(3))) short4_t lds_short4;
    typedef __attribute__((address_space(3))) char lds_char;
    lds_char *const dl = (lds_char *)da + ((lane >> 4) & 1) * 32 + (s16 & 3) * 8;
    const int lrow = wave * 8 + 32 * h;
    const long long c0 = (long long)blockIdx.x * chunk_len, c1 = min(c0 + chunk_len, total);
    uint4_t ua[R * 4 / 256];
    float uw[9], uedge = 0.f;  // windows' element tid, and the two past R of window tid / 2
    auto load = [&](long long s) {
        const int live = (int)min((long long)R, c1 - s);
#pragma unroll
        for (int k = 0; k < R * 4 / 256; ++k) {
            ua[k] = ((const uint4_t *)(dout + s * C))[min(tid + k * 256, live * 4 - 1)];
            if (tid + k * 256 >= live * 4) ua[k] = uint4_t{0, 0, 0, 0};
        }
        // element j of window (dz, dy) is row s + (dz ny + dy) nx - 1 + j; rows outside are never used
        auto at = [&](int w, int j) {
            const long long g = s + ((long long)(w / 3 - 1) * ny + (w % 3 - 1)) * nx - 1 + j;
            return x[min(max(g, 0LL), total - 1)];
        };
#pragma unroll
        for (int w = 0; w < 9; ++w) uw[w] = at(w, tid);
        if (tid < 18) uedge = at(tid / 2, R + tid % 2);
    };
    floatx16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    float bsum = 0.f;
    load(c0);
    // this thread's row: its voxel, advanced by R rows per sub-block
    const long long l0 = (c0 + tid) / nx, p0 = l0 / ny;
    int vx = (int)(c0 + tid - l0 * nx), vy = (int)(l0 - p0 * ny), vz = (int)(p0 % nz);
    const int sx = R % nx, sy = R / nx % ny, sz = (int)((long long)R / nx / ny % nz);
#pragma unroll 1
    for (long long s = c0; s < c1; s += R) {
        const int live = (int)min((long long)R, c1 - s);
#pragma unroll
        for (int k = 0; k < R * 4 / 256; ++k) da[tid + k * 256] = ua[k];
#pragma unroll
        for (int w = 0; w < 9; ++w) win[w][tid] = uw[w];
        if (tid < 18) win[tid / 2][R + tid % 2] = uedge;
        near[tid] = (uint8_t)((tid < live ? 1 : 0) | (vx > 0 ? 2 : 0) | (vx < nx - 1 ? 4 : 0) | (vy > 0 ? 8 : 0) |
                              (vy < ny - 1 ? 16 : 0) | (vz > 0 ? 32 : 0) | (vz < nz - 1 ? 64 : 0));
        vx += sx;
        vy += sy;
        vz += sz;
        if (vx >= nx) {
            vx -= nx;
            ++vy;
        }
        if (vy >= ny) {
            vy -= ny;
            ++vz;
        }
        if (vz >= nz) vz -= nz;
        __syncthreads();
        if (s + R < c1) load(s + R);
        bsum = bias_rows(bsum, (const uint16_t *)da, live);
#pragma unroll
        for (int st = 0; st < R / 64; ++st) {
            typedef short short8_t __attribute__((ext_vector_type(8)));
            const int r0 = 64 * st + lrow;
            short4_t af[2];
#pragma unroll
            for (int p = 0; p < 2; ++p)
                af[p] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4 *)(dl + (r0 + (s16 >> 2) + 4 * p) * (C * 2)));
            const uint2_t f = *(const uint2_t *)(near + r0);
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                v[j] = xw[r0 + j];
                if (((f[j / 4] >> (8 * (j % 4))) & need) != need) v[j] = 0.f;
            }
            const uint4_t b{pack_bf(v[0], v[1]), pack_bf(v[2], v[3]), pack_bf(v[4], v[5]), pack_bf(v[6], v[7])};
            const short8_t a = __builtin_shufflevector(af[0], af[1], 0, 1, 2, 3, 4, 5, 6, 7);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), acc, 0, 0, 0);
        }
        __syncthreads();
    }
    float *red = (float *)da;
    bias_partial(bsum, red, bpart + (size_t)blockIdx.x * C);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 16; ++r) red[wave * C * C + (8 * (r / 4) + 4 * h + r % 4) * C + i] = acc[r];
    __syncthreads();
    float *dst = part + (size_t)blockIdx.x * (C * C);
    for (int e = tid; e < C * C; e += 256)
        dst[e] = ((red[e] + red[C * C + e]) + red[2 * C * C + e]) + red[3 * C * C + e];
}

// bf16 weights of one layer: forward order wf[t][n][k] = W[t][n][k] and the
// data-gradient order wb[t][k][n] = W[26 - t][n][k]; either may be NULL
__device__ __forceinline__ void put_weight(int idx, float v, uint16_t *__restrict__ wf, uint16_t *__restrict__ wb) {
    const int t = idx / (C * C), n = (idx / C) % C, k = idx % C;
    const uint16_t h = f2bf(v);
    if (wf) wf[idx] = h;
    if (wb) wb[((size_t)(TAPS - 1 - t) * C + k) * C + n] = h;
}

__global__ void kc_prep_weights(const float *__restrict__ W, uint16_t *__restrict__ wf, uint16_t *__restrict__ wb) {
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx < TAPS * C * C) put_weight(idx, W[idx], wf, wb);
}

// The minibatch of step `step`: sample s of the batch is training pair
// pick[step * batch + s]
__global__ __launch_bounds__(256) void kc_pick(int V, int batch, int step, const int *__restrict__ pick,
                                               const float *__restrict__ data_in, const float *__restrict__ data_t,
                                               const float *__restrict__ data_tn, float *__restrict__ xin,
                                               float *__restrict__ tgt, float *__restrict__ tn) {
    const int s = blockIdx.y, p = pick[(size_t)step * batch + s];
    const float *in = data_in + (size_t)p * V, *t = data_t + (size_t)p * V;
    for (int v = blockIdx.x * 256 + threadIdx.x; v < V; v += gridDim.x * 256) {
        xin[(size_t)s * V + v] = in[v];
        tgt[(size_t)s * V + v] = t[v];
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) tn[s] = data_tn[p];
}

// round an FP32 tensor to bf16
__global__ void kc_to_bf16(long long len, const float *__restrict__ a, uint16_t *__restrict__ b) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < len; i += (long long)gridDim.x * blockDim.x)
        b[i] = f2bf(a[i]);
}

// ---------------------------------------------------------------------------
// Loss and its gradient.  Sample s of the batch has prediction z[g] (g in its
// V rows) and target tgt[s*V + v] with tn[s] = ||tgt_s||^2:
//   loss = (1/B) sum_s ||z_s - tgt_s||^2 / tn[s]
//   dz[g] = 2 (z - tgt) / (B tn[s]), rounded to bf16.
// part[s * nblk + block] = the block's share of ||z_s - tgt_s||^2.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void kc_loss(int V, int B, int nblk, const float *__restrict__ z,
                                               const float *__restrict__ tgt, const float *__restrict__ tn,
                                               float *__restrict__ dz, float *__restrict__ part) {
    __shared__ float red[256];
    const int s = blockIdx.y;
    float acc = 0.f;
    const float scale = 2.f / ((float)B * tn[s]);
    for (int v = blockIdx.x * 256 + threadIdx.x; v < V; v += nblk * 256) {
        const long long g = (long long)s * V + v;
        const float d = z[g] - tgt[g];
        acc += d * d;
        dz[g] = bf2f(f2bf(scale * d));
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if (threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[(size_t)s * nblk + blockIdx.x] = red[0];
}

// the bf16 weights of the layers, which the optimiser keeps up to date
constexpr int MAX_LAYERS = 4;
struct LayerWeights {
    uint16_t *wf[MAX_LAYERS], *wb[MAX_LAYERS];
};

// Adam (Kingma and Ba, 2015) on FP32 master parameters; mask[i] == 0 keeps a
// padded parameter at zero.  layer_len parameters per layer, weights first.
__global__ void kc_adam(int n, float *__restrict__ p, const float *__restrict__ g, float *__restrict__ m,
                        float *__restrict__ v, const uint8_t *__restrict__ mask, float lr, float b1, float b2,
                        float eps, float c1, float c2, int layer_len, LayerWeights lw) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || !mask[i]) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float pi = p[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    p[i] = pi;
    const int l = i / layer_len, j = i % layer_len;
    if (j < TAPS * C * C) put_weight(j, pi, lw.wf[l], lw.wb[l]);
}

}  // namespace cnn
}  // namespace plsqr
