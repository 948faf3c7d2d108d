// 3D U-Net building blocks on the MFMA cores (BF16 operands, FP32 accumulate).
//
// No reference counterpart (LibGeoDecomp has no learned initial guess).
// Conventions:
//  * activations are channels-last BF16 cubes: element (z,y,x,c) of an n^3
//    tensor with channel stride `ld` and channel offset `off` lives at
//    ((z*n + y)*n + x)*ld + off + c; concatenation is two producers writing
//    disjoint channel ranges of one buffer;
//  * convolution weights are BF16 [cout][Kp] with k = tap*cin + ci,
//    tap = (dz+1)*9 + (dy+1)*3 + (dx+1) for 3x3x3 (tap 0 for 1x1x1), K padded
//    with zeros to Kp = roundup(taps*cin, 32); zero padding at the volume
//    faces ("same" convolution);
//  * a convolution is an implicit GEMM Y[v][co] = sum_k A(v,k) W[co][k] with
//    A(v,k) = X[v + tap(k)][ci(k)], evaluated 16 voxels x 16 channels x 32 k
//    at a time by v_mfma_f32_16x16x32_bf16.
// dgrad is the same kernel with flipped, transposed weights; wgrad reduces
// dY^T X over voxels with the same instruction and a fixed-order reduction.
#include "lgdhip_internal.h"

#include <hip/hip_bf16.h>

#include <algorithm>
#include <cmath>

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16;

// round-to-nearest-even FP32 -> BF16 (finite values)
__device__ __forceinline__ u16 f2bf(float f) {
    uint32_t u = __float_as_uint(f);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (u16)(u >> 16);
}
__device__ __forceinline__ float bf2f(u16 h) { return __uint_as_float((uint32_t)h << 16); }

union Frag {
    bf16x8 v;
    uint4 q;
    u16 h[8];
};

__device__ __forceinline__ void tap_offset(int tap, int ksize, int &dz, int &dy, int &dx) {
    if (ksize == 1) {
        dz = dy = dx = 0;
    } else {
        dz = tap / 9 - 1;
        dy = (tap / 3) % 3 - 1;
        dx = tap % 3 - 1;
    }
}

// A fragment: 8 consecutive k of voxel (z, y, x) -- one 16-byte load when
// the 8 k share a tap (cin % 8 == 0); for even cin with even stride and
// offset, 4 loads of two channels (k and k+1 always share a tap there);
// else element-wise.  The fragment's values are the same in every case.
__device__ __forceinline__ Frag load_a(const u16 *__restrict__ X, int n, int ld, int off, int cin, int ksize,
                                       int z, int y, int x, int k0, int K) {
    Frag f;
    f.q = make_uint4(0, 0, 0, 0);
    if ((cin & 7) == 0) {
        if (k0 < K) {
            const int tap = k0 / cin, ci = k0 % cin;
            int dz, dy, dx;
            tap_offset(tap, ksize, dz, dy, dx);
            const int zz = z + dz, yy = y + dy, xx = x + dx;
            if ((unsigned)zz < (unsigned)n && (unsigned)yy < (unsigned)n && (unsigned)xx < (unsigned)n) {
                f.q = *reinterpret_cast<const uint4 *>(X + ((int64_t)((zz * n + yy) * n + xx)) * ld + off + ci);
            }
        }
    } else if ((cin & 1) == 0 && ((ld | off) & 1) == 0 && ((uintptr_t)X & 3) == 0) {
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
            const int k = k0 + e;  // even: channels ci, ci + 1 of one tap
            if (k < K) {
                const int tap = k / cin, ci = k % cin;
                int dz, dy, dx;
                tap_offset(tap, ksize, dz, dy, dx);
                const int zz = z + dz, yy = y + dy, xx = x + dx;
                if ((unsigned)zz < (unsigned)n && (unsigned)yy < (unsigned)n && (unsigned)xx < (unsigned)n) {
                    const uint32_t pr = *reinterpret_cast<const uint32_t *>(
                        X + ((int64_t)((zz * n + yy) * n + xx)) * ld + off + ci);
                    f.h[e] = (u16)(pr & 0xFFFFu);
                    f.h[e + 1] = (u16)(pr >> 16);
                }
            }
        }
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int k = k0 + e;
            if (k < K) {
                const int tap = k / cin, ci = k % cin;
                int dz, dy, dx;
                tap_offset(tap, ksize, dz, dy, dx);
                const int zz = z + dz, yy = y + dy, xx = x + dx;
                if ((unsigned)zz < (unsigned)n && (unsigned)yy < (unsigned)n && (unsigned)xx < (unsigned)n)
                    f.h[e] = X[((int64_t)((zz * n + yy) * n + xx)) * ld + off + ci];
            }
        }
    }
    return f;
}

constexpr int kMaxNTiles = 12;  // cout up to 192 (the dgrad of a 192-channel concat input)

// One wave: MT x 16 consecutive voxels (linear order, any n) times NT cout
// tiles of 16, the tiles [g NT, g NT + NT) of cout group g (groups split the
// cout tiles when the voxel tiles alone give too few waves; consecutive waves
// are the groups of one voxel range, so they share its A fragments in
// cache).  Each k step loads MT A fragments and NT B fragments for MT x NT
// MFMAs: the weight fragments are shared by the MT voxel tiles.  Every output
// accumulates over k in the same order whatever the split.
template <int NT, int MT>
__global__ __launch_bounds__(256) void conv3d_fwd_mfma(const u16 *__restrict__ X, int n, int ldx, int offx, int cin,
                                                       int ksize, const u16 *__restrict__ W, int Kp,
                                                       const float *__restrict__ bias, int cout, u16 *Y, int ldy,
                                                       int offy, float *Y32, int ld32, int relu, int accumulate,
                                                       int groups) {
    const int lane = threadIdx.x & 63;
    const int64_t wave_id = (int64_t)blockIdx.x * 4 + threadIdx.x / 64;
    const int tile0 = (int)(wave_id % groups) * NT;  // first cout tile of this wave
    const int64_t wave = wave_id / groups;
    const int64_t nvox = (int64_t)n * n * n;
    const int64_t v0 = wave * 16 * MT;
    if (v0 >= nvox) return;
    const int i = lane & 15;   // voxel of the A rows / channel of the B columns
    const int kq = lane >> 4;  // which 8 of the 32 k
    const int K = (ksize == 1 ? 1 : 27) * cin;
    // this lane's A voxel in each of the MT tiles
    bool a_ok[MT];
    int ax[MT], ay[MT], az[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int64_t va = v0 + m * 16 + i;
        a_ok[m] = va < nvox;
        ax[m] = (int)(va % n);
        ay[m] = (int)((va / n) % n);
        az[m] = (int)(va / ((int64_t)n * n));
    }

    f32x4 acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};

    for (int kc = 0; kc < Kp; kc += 32) {
        const int k0 = kc + 8 * kq;
        Frag a[MT], b[NT];
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            a[m].q = make_uint4(0, 0, 0, 0);
            if (a_ok[m]) a[m] = load_a(X, n, ldx, offx, cin, ksize, az[m], ay[m], ax[m], k0, K);
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int co = (tile0 + t) * 16 + i;
            b[t].q = make_uint4(0, 0, 0, 0);
            if (co < cout) b[t].q = *reinterpret_cast<const uint4 *>(W + (int64_t)co * Kp + k0);
        }
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int t = 0; t < NT; ++t)
                acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[m].v, b[t].v, acc[m][t], 0, 0, 0);
    }
    // D[r][c] in lane c + 16*(r/4), element r%4: voxel v0 + 16m + 4*(lane/16) + e, channel (tile0+t)*16 + lane%16
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int co = (tile0 + t) * 16 + i;
        if (co >= cout) continue;
        const float bv = bias ? bias[co] : 0.0f;
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int64_t v = v0 + m * 16 + 4 * kq + e;
                if (v >= nvox) continue;
                float r = acc[m][t][e] + bv;
                if (relu) r = r > 0.0f ? r : 0.0f;
                if (Y) {
                    u16 *p = Y + v * ldy + offy + co;
                    if (accumulate) r += bf2f(*p);
                    *p = f2bf(r);
                }
                if (Y32) Y32[v * ld32 + co] = r;
            }
    }
}

// LDS-staged implicit GEMM for 3x3x3 convolutions with at most 32 output
// channels (NT = 1 or 2 tiles of 16): the U-Net's 128^3 and 64^3 levels,
// where a wave's A fragments (16 voxels x 32 k) feed only NT MFMAs each, so
// fetching them from global memory per MFMA is bound by L1 delivery.
// A work-group computes a 16 x 8 x TZ block of output voxels (TZ = 8 / NT);
// each of its 4 waves owns RT = 16 / NT rows of 16 voxels along x.  The
// input channels are taken 8 at a time (a "group"): the block's input tile
// with its one-voxel halo, (16+2) x (8+2) x (TZ+2) voxels x 8 channels, is
// staged in LDS (two buffers: the next group's global loads are in flight
// while the current one is computed), zeros outside the volume giving the
// faces' zero padding.  A group's 27 taps x 8 channels are seven k steps of
// v_mfma_f32_16x16x32_bf16: in step j, lane group q (lanes 16q..16q+15)
// holds tap 4j + q (the 28th tap is zero), so every A fragment is one
// 16-byte LDS read per lane, voxel (x0 + i + dx, y + dy, z + dz).  The
// group's weight fragments (7 x NT) are loaded once and used for all RT
// rows.  The k order (group-major, then tap) differs from
// conv3d_fwd_mfma's; each output is still one FP32 accumulation of the same
// BF16 products.
constexpr int kLdsTX = 16, kLdsTY = 8;
// 16 zero bytes in device memory: the source of loads that would fall
// outside the volume (or past cout), so no load needs a guard or a select.
// Loads go through global-address-space pointers (global_load, counted by
// vmcnt only; a generic pointer would give flat loads, which LDS waits
// would also wait for).
__device__ __align__(16) const unsigned int kZero16[4] = {0u, 0u, 0u, 0u};
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef const u32x4 __attribute__((address_space(1))) *gq_ptr;
typedef const u16 __attribute__((address_space(1))) *gh_ptr;
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef const u32x2 __attribute__((address_space(1))) *gd_ptr;
__device__ __forceinline__ uint4 load_global16(gh_ptr p) {
    const u32x4 v = *(gq_ptr)p;
    return make_uint4(v.x, v.y, v.z, v.w);
}

__device__ __forceinline__ uint2 load_global8(gh_ptr p) {
    const u32x2 v = *(gd_ptr)p;
    return make_uint2(v.x, v.y);
}

// IN: how the input is staged -- kInVec, 16-byte loads (cin % 8 == 0);
// kInMasked, 16-byte loads of a row whose channels past cin (< 8) are
// another tensor's or padding and are zeroed; kInElem, one load per
// channel.  VST: the output tile goes out as 16-byte stores through LDS
// (plain BF16 output of full cout tiles, no accumulation, no FP32 copy).
constexpr int kInElem = 0, kInVec = 1, kInMasked = 2;

template <int NT, int IN, bool VST>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void conv3d_fwd_lds(const u16 *__restrict__ X, int n, int ldx, int offx, int cin,
                                                      const u16 *__restrict__ W, int Kp,
                                                      const float *__restrict__ bias, int cout, u16 *Y, int ldy,
                                                      int offy, float *Y32, int ld32, int relu, int accumulate,
                                                      int bx, int by) {
    constexpr int TZ = 8 / NT;                // output planes per block
    constexpr int RT = 16 / NT;               // rows per wave: 8 y rows x TZ / 4 planes
    constexpr int SX = kLdsTX + 2, SY = kLdsTY + 2, SZ = TZ + 2;
    constexpr int SV = SX * SY * SZ;          // staged voxels
    constexpr int PER = (SV + 255) / 256;     // staging loads per thread
    __shared__ uint4 tile[2][SV];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int i = lane & 15, q = lane >> 4;
    int b = blockIdx.x;
    const int x0 = (b % bx) * kLdsTX;
    b /= bx;
    const int y0 = (b % by) * kLdsTY;
    const int z0 = (b / by) * TZ;
    const int groups = (cin + 7) / 8;

    // staged voxel p of this thread: its element offset in X (0 and a zero
    // mask outside the volume, so every load is issued unconditionally and
    // all of a thread's loads are in flight together)
    int64_t soff[PER];
    bool sok[PER];
#pragma unroll
    for (int p = 0; p < PER; ++p) {
        const int sv = tid + 256 * p;
        const int xx = x0 + sv % SX - 1, yy = y0 + (sv / SX) % SY - 1, zz = z0 + sv / (SX * SY) - 1;
        sok[p] = sv < SV && (unsigned)xx < (unsigned)n && (unsigned)yy < (unsigned)n && (unsigned)zz < (unsigned)n;
        soff[p] = sok[p] ? (((int64_t)zz * n + yy) * n + xx) * ldx : 0;
    }
    uint4 stage[PER];
    const gh_ptr zero = (gh_ptr)(const void *)kZero16;
    const gh_ptr xg = (gh_ptr)X;
    auto stage_load = [&](int c) {
        const gh_ptr base = xg + offx + 8 * c;
#pragma unroll
        for (int p = 0; p < PER; ++p) {
            Frag f;
            if (IN != kInElem) {
                f.q = load_global16(sok[p] ? base + soff[p] : zero);
                if (IN == kInMasked) {
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (e >= cin) f.h[e] = 0;
                }
            } else {
                // channels beyond cin (and voxels outside) read zeros
#pragma unroll
                for (int e = 0; e < 8; ++e) f.h[e] = *(sok[p] && 8 * c + e < cin ? base + soff[p] + e : zero);
            }
            stage[p] = f.q;
        }
    };
    auto stage_store = [&](int buf) {
#pragma unroll
        for (int p = 0; p < PER; ++p) {
            const int sv = tid + 256 * p;
            if (sv < SV) tile[buf][sv] = stage[p];
        }
    };

    // this lane group's tap of each k step, as an offset in the staged tile
    // relative to the row's first voxel (x0 - 1, y - 1, z - 1)
    int toff[7];
    bool tok[7];
#pragma unroll
    for (int j = 0; j < 7; ++j) {
        const int tap = 4 * j + q;
        tok[j] = tap < 27;
        int dz, dy, dx;
        tap_offset(tok[j] ? tap : 13, 3, dz, dy, dx);
        toff[j] = ((dz + 1) * SY + (dy + 1)) * SX + (dx + 1) + i;
    }

    f32x4 acc[RT][NT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[r][t] = f32x4{0.f, 0.f, 0.f, 0.f};

    // a group's weight fragments: channels 8c..8c+7 of tap 4j + q for output
    // channel t * 16 + i (zero for the 28th tap, channels past cout or cin)
    Frag bf[7][NT];
    auto load_b = [&](int c) {
#pragma unroll
        for (int j = 0; j < 7; ++j)
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const int co = t * 16 + i;
                const bool ok = tok[j] && co < cout;
                const gh_ptr src = (gh_ptr)W + (int64_t)co * Kp + (4 * j + q) * cin + 8 * c;
                if (IN == kInVec) {
                    bf[j][t].q = load_global16(ok ? src : zero);
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e) bf[j][t].h[e] = *(ok && 8 * c + e < cin ? src + e : zero);
                }
            }
    };

    // Software pipeline over the groups.  Loads complete in issue order
    // (vmcnt), so each group's loads are issued after the ones it waits for
    // last: the staged input of group c + 1 goes out first, the MFMAs of
    // group c then need only the weights loaded in the previous iteration;
    // the weights of group c + 1 go out after the MFMAs, and writing the
    // staged input waits only for the older staging loads.
    stage_load(0);
    load_b(0);
    stage_store(0);
    __syncthreads();
    for (int c = 0; c < groups; ++c) {
        const int cur = c & 1;
        // the next group's loads are issued unconditionally (the last group
        // re-reads its own, never stored), so the wait counts are the same on
        // every iteration and exact
        const int cn = c + 1 < groups ? c + 1 : c;
        stage_load(cn);  // in flight during the MFMAs below
        // k step outermost: consecutive MFMAs update different rows'
        // accumulators, so none waits for the previous one's result
        // (the 28th tap's zero weights make its A values irrelevant: it reads
        // the block's centre tap, always inside the staged tile)
#pragma unroll
        for (int j = 0; j < 7; ++j) {
            Frag a[RT];  // all rows' fragments of this k step in flight together
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                const int yl = r % 8, zl = wave * (TZ / 4) + r / 8;
                a[r].q = tile[cur][(zl * SY + yl) * SX + toff[j]];
            }
#pragma unroll
            for (int r = 0; r < RT; ++r)
#pragma unroll
                for (int t = 0; t < NT; ++t)
                    acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[r].v, bf[j][t].v, acc[r][t], 0, 0, 0);
        }
        // schedule: kLdsAhead fragment reads in flight ahead of the MFMAs
        // that consume them (the compiler alone keeps two, and each MFMA
        // then waits out an LDS latency)
        constexpr int kReads = 7 * RT, kLdsAhead = 8;
        __builtin_amdgcn_sched_group_barrier(0x100, kLdsAhead, 0);
        lgdhip::static_for<0, kReads - kLdsAhead>([&](auto) {
            __builtin_amdgcn_sched_group_barrier(0x008, NT, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        });
        __builtin_amdgcn_sched_group_barrier(0x008, NT * kLdsAhead, 0);
        load_b(cn);
        if (c + 1 < groups) stage_store(cur ^ 1);
        __syncthreads();
    }
    // D[r][c] in lane c + 16 (r / 4), element r % 4: voxel x0 + 4q + e of the
    // row, channel t * 16 + i
    if (VST) {
        // through LDS (the staging buffers are free after the last barrier):
        // [voxel of the block][16 NT channels] BF16, then 16-byte stores
        constexpr int CH = 16 * NT;
        u16 *otile = reinterpret_cast<u16 *>(&tile[0][0]);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int co = t * 16 + i;
            const float bv = bias ? bias[co] : 0.0f;
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                const int vt = ((wave * (TZ / 4) + r / 8) * 8 + r % 8) * 16 + 4 * q;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float o = acc[r][t][e] + bv;
                    if (relu) o = o > 0.0f ? o : 0.0f;
                    otile[(vt + e) * CH + co] = f2bf(o);
                }
            }
        }
        __syncthreads();
        constexpr int CHUNKS = 16 * 8 * TZ * CH / 8;  // 16-byte pieces of the block
#pragma unroll
        for (int k = tid; k < CHUNKS; k += 256) {
            const int vt = k / (CH / 8), part = k % (CH / 8);
            const int x = x0 + vt % 16, y = y0 + (vt / 16) % 8, z = z0 + vt / 128;
            if (x < n && y < n && z < n) {
                const int64_t v = ((int64_t)z * n + y) * n + x;
                *reinterpret_cast<uint4 *>(Y + v * ldy + offy + 8 * part) =
                    *reinterpret_cast<const uint4 *>(otile + vt * CH + 8 * part);
            }
        }
        return;
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int co = t * 16 + i;
        if (co >= cout) continue;
        const float bv = bias ? bias[co] : 0.0f;
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            const int y = y0 + r % 8, z = z0 + wave * (TZ / 4) + r / 8;
            if (y >= n || z >= n) continue;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int x = x0 + 4 * q + e;
                if (x >= n) continue;
                const int64_t v = ((int64_t)z * n + y) * n + x;
                float o = acc[r][t][e] + bv;
                if (relu) o = o > 0.0f ? o : 0.0f;
                if (Y) {
                    u16 *pp = Y + v * ldy + offy + co;
                    if (accumulate) o += bf2f(*pp);
                    *pp = f2bf(o);
                }
                if (Y32) Y32[v * ld32 + co] = o;
            }
        }
    }
}

// all ones in the halves of a word of two BF16 values that are positive
__device__ __forceinline__ uint32_t positive_halves(uint32_t w) {
    return (__uint_as_float(w << 16) > 0.0f ? 0xFFFFu : 0u) |
           (__uint_as_float(w & 0xFFFF0000u) > 0.0f ? 0xFFFF0000u : 0u);
}

// Z-marching LDS convolution for 3x3x3 layers with cin = 8 G input channels (G
// <= 6; G = 1 also takes cin < 8 rows, see IN) and slices of NT x 16 output
// channels.  A work-group owns a 16 x 8 column of output voxels and one slice and
// marches z over a chunk of planes.  Input planes (18 x 10 voxels with their
// halo, all cin channels) pass through a ring of 4 LDS slots: output plane z
// reads input planes z-1, z, z+1 while plane z+2 is written into the fourth
// slot; up to two planes' loads are in flight in registers, so a load has a whole
// step to arrive.  Every input voxel is fetched once per column and slice, whole
// channel rows together (the tile kernel above takes the channels 8 at a time,
// re-reading each voxel's row G times).  Wave w computes output rows y0 + 2w and
// y0 + 2w + 1 of each plane.  The G x 7 x NT weight fragments of the lane stay in
// registers for the whole march; a plane step is bound by the LDS reads of the
// input fragments, so each feeds NT products.  Work-groups run in XCD order,
// slices of a column together: neighbouring columns' halos come from one L2.
//
// The k order is that of the kernel that takes the layer when this one does not
// (accumulation, unaligned rows), so a layer's result has the same bits either
// way, with two exceptions that differ by roundings of the FP32 sums: plain
// launches of 2 to 6 groups and more than 32 output channels on 96^3 and larger
// (kZmGroupOrderN), and masked rows with more than 32 output channels, which
// conv3d_fwd_mfma takes otherwise.  SPLIT = 0: conv3d_fwd_lds's, group-major, 4 taps of one group per step.
// SPLIT = 1: conv3d_fwd_gemm's, the weights' tap-major rows, 4 groups (of one
// tap or two) per step.  SPLIT = 2: the same in conv3d_fwd_gemm's two slices of
// its stages, each summed from zero and then added.
//
// MASK: outputs whose activation A (rows of lda elements) is not positive are
// zeroed: the ReLU backward of the layer that made the tensor this one is the
// gradient of, without a pass of its own (a training step at 128^3 took 2108 us
// with these passes, 1997 us with the masks taken along here, in conv1x1_from1
// and in the resampling gradients).
//
// Measured (us; the launch this one replaces in brackets: one 16-channel slice
// per launch with the outputs re-tiled in LDS; the GEMM-tiled kernel and its
// reduction; the LDS-tile kernel): 128^3 16 -> 16 41 [48], 3 -> 16 36 [47], 48 ->
// 16 114 [127], 16 -> 48 102 [147], 32 -> 32 115 [145]; 100^3 64 -> 16 168 [tile
// 237]; 64^3 32 -> 96 54 [GEMM 143], 64 -> 64 92 [GEMM 124], 32 -> 32 21.5 [tile
// 24.6]; 60^3 16 -> 16 11 [34], 32 -> 32 20 [GEMM 67], 48 -> 32 33 [GEMM 89]; 32^3
// 32 -> 64 9.5 [GEMM 25], 64 -> 64 21 [GEMM 31]; 16^3 16 -> 16 6 [18].
// work-groups per CU (and waves per SIMD), by registers and, from 7 groups on, LDS
constexpr int zm_waves(int g, int nt) { return g * nt <= 2 ? 3 : (g * nt <= 6 ? 2 : 1); }
// planes in flight: one where the weight fragments leave no registers for two
constexpr int zm_ahead(int g, int nt) { return g * nt == 5 || g * nt == 6 ? 1 : 2; }
// k steps of 32, and the one a SPLIT = 2 launch's second slice begins with
constexpr int zm_steps(int g, int split) { return split ? (27 * g + 3) / 4 : 7 * g; }
constexpr int zm_second(int g) { return (zm_steps(g, 2) + 1) / 2 / 2 * 2; }
// fragment reads in flight (at 6 groups the weights leave room for three: 48 ->
// 16 at 128^3 133 us with six, 115 with three; in tap-major order for two: 48 ->
// 32 at 60^3 38.6 us with three, 32.6 with two)
constexpr int zm_reads(int g, int split) { return g == 6 ? (split ? 2 : 3) : 6; }

template <int G, int IN, int NT, int SPLIT, bool MASK>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(zm_waves(G, NT), zm_waves(G, NT)))) void
conv3d_fwd_zm(const u16 *__restrict__ X, int n, int ldx, int offx, int cin, const u16 *__restrict__ W, int Kp,
              const float *__restrict__ bias, u16 *Y, int ldy, int offy, float *Y32, int ld32, int relu,
              const u16 *__restrict__ A, int lda, int offa, int bx, int by, int slices, int zchunk, unsigned groups,
              unsigned per) {
    constexpr int SX = 18, SY = 10, PV = SX * SY;  // staged voxels per plane
    constexpr int CHUNKS = PV * G;                 // 16-byte pieces per plane
    constexpr int PER = (CHUNKS + 255) / 256;
    constexpr int OC = 16 * NT;  // output channels of the slice
    // [slot][group][voxel]; tap-major steps read up to 4 groups at one voxel
    // offset, 256 bytes apart modulo the banks where the groups' stride is padded
    // (60^3 32 -> 32 21.4 us unpadded, 20.0 padded, 48 -> 32 36.7 and 32.8; from 7
    // groups on the staging writes conflict instead and it lost 5 %)
    constexpr int PS = SPLIT && G <= 6 ? (PV + 15) / 16 * 16 : PV;
    // the last SX + 1 pieces of a slot stay zero: what a lane past the last tap
    // reads (its weights are zero, but zero times an infinite activation is NaN)
    constexpr int ZERO = PS * G;
    __shared__ uint4 ring[4][ZERO + SX + 1];
    unsigned b = lgdhip::xcd_tile(blockIdx.x, per, true);
    if (b >= groups) return;  // whole work-group, before any barrier
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int i = lane & 15, q = lane >> 4;
    const int slice = (int)(b % slices);
    b /= slices;
    const int x0 = (int)(b % bx) * 16;
    b /= bx;
    const int y0 = (int)(b % by) * 8;
    const int z0 = (int)(b / by) * zchunk;
    const int zend = min(z0 + zchunk, n);
    W += (int64_t)slice * OC * Kp;
    offy += slice * OC;
    offa += slice * OC;

    const gh_ptr zero = (gh_ptr)(const void *)kZero16;
    const gh_ptr xg = (gh_ptr)X + offx;
    // this thread's pieces of a plane: voxel sv = k / G, group g = k % G
    // (consecutive threads read consecutive 16 bytes of the voxels' rows)
    int pofs[PER];   // element offset within a plane's (x, y) footprint
    bool pok[PER];
#pragma unroll
    for (int p = 0; p < PER; ++p) {
        const int k = tid + 256 * p;
        const int sv = k / G, g = k % G;
        const int xx = x0 + sv % SX - 1, yy = y0 + sv / SX - 1;
        pok[p] = k < CHUNKS && (unsigned)xx < (unsigned)n && (unsigned)yy < (unsigned)n;
        pofs[p] = pok[p] ? (yy * n + xx) * ldx + 8 * g : 0;
    }
    constexpr int PF = zm_ahead(G, NT);
    uint4 stage[PF][PER];
    auto plane_load = [&](int set, int z) {
        const bool zok = (unsigned)z < (unsigned)n;
        const gh_ptr base = xg + (int64_t)(zok ? z : 0) * n * n * ldx;
#pragma unroll
        for (int p = 0; p < PER; ++p) {
            Frag f;
            f.q = load_global16(pok[p] && zok ? base + pofs[p] : zero);
            if (IN == kInMasked) {
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (e >= cin) f.h[e] = 0;
            }
            stage[set][p] = f.q;
        }
    };
    auto plane_store = [&](int set, int slot) {
#pragma unroll
        for (int p = 0; p < PER; ++p) {
            const int k = tid + 256 * p;
            if (k < CHUNKS) ring[slot][(k % G) * PS + k / G] = stage[set][p];
        }
    };

    // A step's fragment reads and weights: lane group q takes tap and group of
    // the step's chunk q (zero weights past the last tap and past cin).  Chunks
    // 4 s .. 4 s + 3 of a tap-major row lie in at most two taps (G >= 2).
    constexpr int STEPS = zm_steps(G, SPLIT);
    auto chunk_of = [&](int st, int &tap, int &g) __attribute__((always_inline)) {
        if (SPLIT) {
            const int t0 = 4 * st / G, t1 = (4 * st + 3) / G;
            tap = t0 == t1 || 4 * st + q < G * t1 ? t0 : t1;
            g = 4 * st + q - G * tap;
        } else {
            tap = 4 * (st % 7) + q;
            g = st / 7;
        }
        const bool ok = tap < 27;
        if (!ok) tap = 13, g = 0;
        return ok;
    };
    Frag bf[STEPS][NT];
#pragma unroll
    for (int j = 0; j < STEPS; ++j)
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            int tap, g;
            const bool ok = chunk_of(j, tap, g);
            const gh_ptr src = (gh_ptr)W + (int64_t)(16 * t + i) * Kp + tap * cin + 8 * g;
            if (IN == kInVec) {
                bf[j][t].q = load_global16(ok ? src : zero);
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) bf[j][t].h[e] = *(ok && e < cin ? src + e : zero);
            }
        }
    // ring offset of row 2 wave, voxel i; group-major steps: this lane group's
    // taps' slot (dz + 1) and voxel offset
    const int vox = 2 * wave * SX + i;
    int tslot[7], toff[7];
#pragma unroll
    for (int j = 0; j < 7; ++j) {
        const int tap = 4 * j + q < 27 ? 4 * j + q : 13;
        tslot[j] = tap / 9;
        toff[j] = tap / 3 % 3 * SX + tap % 3 + vox;
    }
    // The products are taken as W X^T, so a lane holds 4 consecutive output
    // channels, 16 t + 4 q .. + 3, of voxel i of its row: 8-byte stores, the 64
    // lanes of a tile 512 contiguous bytes (at 16 channels).
    float bv[NT][4];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) bv[t][e] = bias ? bias[slice * OC + 16 * t + 4 * q + e] : 0.0f;
    const bool xin = x0 + i < n;
    bool rin[2];  // the lane's output voxel of each row is inside
    int vofs[2];  // its index within a plane
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        rin[r] = xin && y0 + 2 * wave + r < n;
        vofs[r] = (y0 + 2 * wave + r) * n + x0 + i;
    }

    if (tid < 4 * (SX + 1)) ring[tid / (SX + 1)][ZERO + tid % (SX + 1)] = make_uint4(0u, 0u, 0u, 0u);
    // prologue: planes z0-1, z0, z0+1 in slots 0..2, the next PF in flight
    plane_load(0, z0 - 1);
    plane_store(0, 0);
    plane_load(0, z0);
    plane_store(0, 1);
    plane_load(0, z0 + 1);
    plane_store(0, 2);
    plane_load(0, z0 + 2);
    if (PF == 2) plane_load(PF - 1, z0 + 3);
    __syncthreads();
    auto step = [&](auto ph_c, int z) __attribute__((always_inline)) {
        constexpr int PH = decltype(ph_c)::value;  // (z - z0) & 1
        const int st = z - z0;
        const int64_t plane = (int64_t)z * n * n;
        // plane z+2 into the free slot, the next PF in flight
        plane_store(PH % PF, (st + 3) & 3);
        plane_load(PH % PF, z + 2 + PF);
        f32x4 acc[2][NT];
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[r][t] = f32x4{0.f, 0.f, 0.f, 0.f};
        uint2 act[2][NT];  // MASK: the outputs' activations
        if (MASK) {
#pragma unroll
            for (int r = 0; r < 2; ++r)
#pragma unroll
                for (int t = 0; t < NT; ++t)
                    act[r][t] = load_global8(
                        (gh_ptr)A + (rin[r] ? (plane + vofs[r]) * lda : 0) + offa + 16 * t + 4 * q);
        }
        f32x4 first[2][NT];  // SPLIT = 2: the first slice's sums
        const uint4 *const slots[3] = {ring[st & 3], ring[(st + 1) & 3], ring[(st + 2) & 3]};
#pragma unroll
        for (int j = 0; j < STEPS; ++j) {
            const uint4 *pl;
            if (SPLIT) {
                // one tap: the lanes differ by their group only; two: by a select
                const int t0 = 4 * j / G, t1 = (4 * j + 3) / G < 27 ? (4 * j + 3) / G : t0;
                const uint4 *p0 = slots[t0 / 9] + (4 * j - G * t0) * PS + t0 / 3 % 3 * SX + t0 % 3;
                const uint4 *p1 = slots[t1 / 9] + (4 * j - G * t1) * PS + t1 / 3 % 3 * SX + t1 % 3;
                if (4 * j + 3 < 27 * G)
                    pl = (t0 == t1 || 4 * j + q < G * t1 ? p0 : p1) + q * PS + vox;
                else  // the last step, all of its chunks of tap 26
                    pl = slots[2] + (q < 27 * G - 4 * j ? (4 * j - 26 * G + q) * PS + 2 * SX + 2 + vox : ZERO);
            } else {
                pl = &ring[(st + tslot[j % 7]) & 3][j / 7 * PS + toff[j % 7]];
                if (j % 7 == 6 && q == 3) pl = &ring[0][ZERO];
            }
            if (SPLIT == 2 && j == zm_second(G)) {
#pragma unroll
                for (int r = 0; r < 2; ++r)
#pragma unroll
                    for (int t = 0; t < NT; ++t) {
                        first[r][t] = acc[r][t];
                        acc[r][t] = f32x4{0.f, 0.f, 0.f, 0.f};
                    }
            }
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                Frag a;
                a.q = pl[r * SX];
#pragma unroll
                for (int t = 0; t < NT; ++t)
                    acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[j][t].v, a.v, acc[r][t], 0, 0, 0);
            }
        }
        // schedule: kReads fragment reads in flight ahead of the products that
        // consume them (the compiler alone keeps about two, and the step then
        // waits out an LDS latency per k step)
        constexpr int kReads = zm_reads(G, SPLIT);
        __builtin_amdgcn_sched_group_barrier(0x100, kReads, 0);
        lgdhip::static_for<0, 2 * STEPS - kReads>([&](auto) {
            __builtin_amdgcn_sched_group_barrier(0x008, NT, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        });
        __builtin_amdgcn_sched_group_barrier(0x008, NT * kReads, 0);
        if (SPLIT == 2) {
#pragma unroll
            for (int r = 0; r < 2; ++r)
#pragma unroll
                for (int t = 0; t < NT; ++t)
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[r][t][e] = first[r][t][e] + acc[r][t][e];
        }
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const int64_t v = plane + vofs[r];
            u16 *out = Y + v * ldy + offy + 4 * q;
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                float o[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    o[e] = acc[r][t][e] + bv[t][e];
                    if (relu) o[e] = o[e] > 0.0f ? o[e] : 0.0f;
                }
                uint2 h = make_uint2(f2bf(o[0]) | (uint32_t)f2bf(o[1]) << 16, f2bf(o[2]) | (uint32_t)f2bf(o[3]) << 16);
                if (MASK) {
                    h.x &= positive_halves(act[r][t].x);
                    h.y &= positive_halves(act[r][t].y);
                }
                if (Y && rin[r]) *reinterpret_cast<uint2 *>(out + 16 * t) = h;
                if (Y32 && rin[r]) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) Y32[v * ld32 + slice * OC + 16 * t + 4 * q + e] = o[e];
                }
            }
        }
        __syncthreads();
    };
    int z = z0;
    for (; z + 1 < zend; z += 2) {
        step(lgdhip::ic<0>{}, z);
        step(lgdhip::ic<1>{}, z + 1);
    }
    if (z < zend) step(lgdhip::ic<0>{}, z);
}

// GEMM-tiled implicit convolution for 3x3x3 layers with cin % 8 == 0 on the
// small levels (n < 64) and for cout > 32: Y[v][co] = sum_k A(v, k) W[co][k]
// over a 64-voxel x 64-channel block per work-group.  k runs in stages of 64
// (eight 8-channel chunks of one or more taps); a stage's A block (64 voxels
// x 64 k, gathered from the channels-last input with zeros outside the
// volume) and B block (64 channels x 64 k of the weights) are staged in LDS,
// double buffered: the next stage's global loads are in flight in registers
// while the current one is computed.  Wave w computes the 32 x 32 quarter
// (voxel half w & 1, channel half w >> 1) as 2 x 2 MFMA tiles, two k steps
// of 32 per stage, every fragment one ds_read_b128 (rows padded to 72
// elements: the 16 rows of a fragment read hit distinct banks).  A block
// reads its A and B data from L2 once instead of once per wave.
// With `slices` > 1 the stage range is split over work-groups (a slice
// each, for small volumes whose 64 x 64 blocks alone leave CUs idle) and
// every slice writes FP32 partials P[slice][v][co]; conv3d_gemm_reduce adds
// them in slice order.  k order: stage-major, then k within the stage (the
// tap-major order of the weights), per slice.
constexpr int kGemmBM = 64, kGemmBN = 64, kGemmBK = 64;
constexpr int kGemmLd = kGemmBK + 8;  // LDS row stride in elements (144 bytes)

template <bool SPLIT>
__global__ __launch_bounds__(256) void conv3d_fwd_gemm(const u16 *__restrict__ X, int n, int ldx, int offx, int cin,
                                                       const u16 *__restrict__ W, int Kp,
                                                       const float *__restrict__ bias, int cout, u16 *Y, int ldy,
                                                       int offy, float *Y32, int ld32, int relu, int accumulate,
                                                       int mblocks, int nblocks, int slices, int stages,
                                                       float *__restrict__ P) {
    __shared__ uint4 lds[2][2][kGemmBM * kGemmLd / 8];  // [buffer][A, B][row * kGemmLd / 8 + chunk]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int i = lane & 15, q = lane >> 4;
    int b = blockIdx.x;
    const int mb = b % mblocks;
    b /= mblocks;
    const int nb = b % nblocks;
    const int slice = b / nblocks;
    const int64_t nvox = (int64_t)n * n * n;
    const int64_t v0 = (int64_t)mb * kGemmBM;
    const int co0 = nb * kGemmBN;
    const int st0 = (int)((int64_t)slice * stages / slices), st1 = (int)((int64_t)(slice + 1) * stages / slices);
    const int K = 27 * cin;

    // loader roles: chunk c = tid + 256 u (u = 0, 1) of the 512 16-byte
    // chunks of each block: row c / 8, k chunk c % 8 (the same for both)
    const int j = tid & 7;
    const gh_ptr zero = (gh_ptr)(const void *)kZero16;
    const gh_ptr xg = (gh_ptr)X + offx;
    int vx[2], vy[2], vz[2];
    bool vok[2];
    const gh_ptr wrow[2] = {(gh_ptr)W + (int64_t)(co0 + (tid >> 3)) * Kp,
                            (gh_ptr)W + (int64_t)(co0 + (tid >> 3) + 32) * Kp};
    const bool cok[2] = {co0 + (tid >> 3) < cout, co0 + (tid >> 3) + 32 < cout};
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int64_t v = v0 + (tid >> 3) + 32 * u;
        vok[u] = v < nvox;
        vx[u] = (int)(v % n);
        vy[u] = (int)((v / n) % n);
        vz[u] = (int)(v / ((int64_t)n * n));
    }
    const float inv_cin = 1.0f / (float)cin;
    uint4 ra[2], rb[2];
    auto load_stage = [&](int st) {
        const int k0 = st * kGemmBK + 8 * j;
        // tap = k0 / cin from a float reciprocal, corrected (k0 < 2^24)
        int tap = (int)((float)k0 * inv_cin);
        tap -= tap * cin > k0;
        tap += (tap + 1) * cin <= k0;
        const int ci = k0 - tap * cin;
        const bool kin = k0 < K;
        int dz, dy, dx;
        tap_offset(kin ? tap : 13, 3, dz, dy, dx);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int zz = vz[u] + dz, yy = vy[u] + dy, xx = vx[u] + dx;
            const bool ok = kin && vok[u] && (unsigned)zz < (unsigned)n && (unsigned)yy < (unsigned)n &&
                            (unsigned)xx < (unsigned)n;
            ra[u] = load_global16(ok ? xg + ((int64_t)(zz * n + yy) * n + xx) * ldx + ci : zero);
            rb[u] = load_global16(cok[u] && k0 < Kp ? wrow[u] + k0 : zero);
        }
    };
    auto store_stage = [&](int buf) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int row = (tid >> 3) + 32 * u;
            lds[buf][0][row * (kGemmLd / 8) + j] = ra[u];
            lds[buf][1][row * (kGemmLd / 8) + j] = rb[u];
        }
    };

    f32x4 acc[2][2];
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int t = 0; t < 2; ++t) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int wm = wave & 1, wn = wave >> 1;
    if (st0 < st1) {
        load_stage(st0);
        store_stage(0);
        __syncthreads();
        for (int st = st0; st < st1; ++st) {
            const int cur = (st - st0) & 1;
            // the next stage's loads go out first (the last stage re-loads
            // its own, never stored, so every iteration waits alike)
            load_stage(st + 1 < st1 ? st + 1 : st);
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                Frag a[2], bf[2];
#pragma unroll
                for (int m = 0; m < 2; ++m)
                    a[m].q = lds[cur][0][(32 * wm + 16 * m + i) * (kGemmLd / 8) + 4 * ks + q];
#pragma unroll
                for (int t = 0; t < 2; ++t)
                    bf[t].q = lds[cur][1][(32 * wn + 16 * t + i) * (kGemmLd / 8) + 4 * ks + q];
#pragma unroll
                for (int m = 0; m < 2; ++m)
#pragma unroll
                    for (int t = 0; t < 2; ++t)
                        acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[m].v, bf[t].v, acc[m][t], 0, 0, 0);
            }
            if (st + 1 < st1) store_stage(cur ^ 1);
            __syncthreads();
        }
    }
    // D[r][c] in lane c + 16 (r / 4), element r % 4: voxel row 4q + e of the
    // tile, channel i
    const int ldp = nblocks * kGemmBN;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int co = co0 + 32 * wn + 16 * t + i;
        const float bv = !SPLIT && bias && co < cout ? bias[co] : 0.0f;
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int64_t v = v0 + 32 * wm + 16 * m + 4 * q + e;
                if (v >= nvox) continue;
                if (SPLIT) {
                    P[((int64_t)slice * nvox + v) * ldp + co] = acc[m][t][e];
                    continue;
                }
                if (co >= cout) continue;
                float r = acc[m][t][e] + bv;
                if (relu) r = r > 0.0f ? r : 0.0f;
                if (Y) {
                    u16 *pp = Y + v * ldy + offy + co;
                    if (accumulate) r += bf2f(*pp);
                    *pp = f2bf(r);
                }
                if (Y32) Y32[v * ld32 + co] = r;
            }
    }
}

// the slices' partials of conv3d_fwd_gemm summed in slice order, then bias,
// ReLU, accumulation and the BF16 / FP32 stores of the unsplit epilogue
__global__ __launch_bounds__(256) void conv3d_gemm_reduce(const float *__restrict__ P, int64_t nvox, int ldp,
                                                          int slices, const float *__restrict__ bias, int cout,
                                                          u16 *Y, int ldy, int offy, float *Y32, int ld32, int relu,
                                                          int accumulate) {
    // a split launch has fewer than 1024 blocks of 64 x 64 outputs, so
    // nvox * cout < 2^22 and 32-bit index arithmetic holds
    const uint32_t idx = blockIdx.x * 256u + threadIdx.x;
    if (idx >= (uint32_t)(nvox * cout)) return;
    const uint32_t v = idx / (uint32_t)cout;
    const int co = (int)(idx - v * (uint32_t)cout);
    float r = 0.0f;
    for (int sl = 0; sl < slices; ++sl) r += P[((int64_t)sl * nvox + v) * ldp + co];
    r += bias ? bias[co] : 0.0f;
    if (relu) r = r > 0.0f ? r : 0.0f;
    if (Y) {
        u16 *pp = Y + (int64_t)v * ldy + offy + co;
        if (accumulate) r += bf2f(*pp);
        *pp = f2bf(r);
    }
    if (Y32) Y32[(int64_t)v * ld32 + co] = r;
}

// 1x1x1 convolution to a single output channel (the U-Net's output layer):
// one thread per voxel, its cin channels in 16-byte loads (cin % 8 == 0), an
// FP32 dot product with the cin weights.  An MFMA tile would compute 16
// output channels to keep one, and the layer is memory bound.
__global__ __launch_bounds__(256) void conv1x1_to1(const u16 *__restrict__ X, int64_t nvox, int ldx, int offx,
                                                   int cin, const u16 *__restrict__ W,
                                                   const float *__restrict__ bias, u16 *Y, int ldy, int offy,
                                                   float *Y32, int ld32, int relu, int accumulate) {
    const int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (v >= nvox) return;
    const u16 *xr = X + v * ldx + offx;
    float acc = 0.0f;
    for (int c = 0; c < cin; c += 8) {
        Frag f, w;
        f.q = *reinterpret_cast<const uint4 *>(xr + c);
        w.q = *reinterpret_cast<const uint4 *>(W + c);
#pragma unroll
        for (int e = 0; e < 8; ++e) acc += bf2f(f.h[e]) * bf2f(w.h[e]);
    }
    float o = acc + (bias ? bias[0] : 0.0f);
    if (relu) o = o > 0.0f ? o : 0.0f;
    if (Y) {
        u16 *pp = Y + v * ldy + offy;
        if (accumulate) o += bf2f(*pp);
        *pp = f2bf(o);
    }
    if (Y32) Y32[v * ld32] = o;
}

// 1x1x1 convolution of a single input channel (the output layer's input
// gradient): y[v][co] = x[v] w[co], 8 output channels per thread.  One product
// each, so the same values as an MFMA tile with 31 zero products, which took
// 52 us at 128^3 x 16 for one pass over 71 MB.  W rows are Kp apart.
__global__ __launch_bounds__(256) void conv1x1_from1(const u16 *__restrict__ X, uint32_t items, int ldx, int offx,
                                                     const u16 *__restrict__ W, int Kp,
                                                     const float *__restrict__ bias, int c8, u16 *__restrict__ Y,
                                                     int ldy, int offy, int relu, const u16 *__restrict__ A, int lda,
                                                     int offa) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= items) return;
    const uint32_t v = i / (uint32_t)c8;
    const int co = 8 * (int)(i - v * (uint32_t)c8);
    const float xv = bf2f(X[(int64_t)v * ldx + offx]);
    Frag f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        float o = xv * bf2f(W[(int64_t)(co + e) * Kp]) + (bias ? bias[co + e] : 0.0f);
        if (relu) o = o > 0.0f ? o : 0.0f;
        f.h[e] = f2bf(o);
    }
    if (A) {  // ReLU backward of the layer that made Y's values, as conv3d_fwd_zm's
        const uint4 a = *reinterpret_cast<const uint4 *>(A + (int64_t)v * lda + offa + co);
        f.q.x &= positive_halves(a.x);
        f.q.y &= positive_halves(a.y);
        f.q.z &= positive_halves(a.z);
        f.q.w &= positive_halves(a.w);
    }
    *reinterpret_cast<uint4 *>(Y + (int64_t)v * ldy + offy + co) = f.q;
}

// Weight gradient of a 1x1x1 layer with one output channel: P[chunk][ci] = sum
// over the chunk's voxels of dY[v] X[v][ci].  Thread (lane, piece) sums 8
// channels of every (256 / c8)-th voxel in FP32; the lanes' sums are added in a
// fixed tree.  One pass over X (an MFMA tile of 16 output channels with element
// gathers took 77 us at 128^3 x 16).
__global__ __launch_bounds__(256) void conv1x1_to1_wgrad(const u16 *__restrict__ X, int64_t nvox, int ldx, int offx,
                                                         const u16 *__restrict__ dY, int ldy, int offy, int c8,
                                                         int Kp, int chunk_vox, float *__restrict__ P) {
    __shared__ float red[256][9];
    const int t = threadIdx.x, lanes = 256 / c8;  // c8 a power of two
    const int piece = t % c8, lane = t / c8;
    const int64_t v0 = (int64_t)blockIdx.x * chunk_vox;
    const int64_t v1 = v0 + chunk_vox < nvox ? v0 + chunk_vox : nvox;
    float s[8] = {};
    for (int64_t v = v0 + lane; v < v1; v += lanes) {
        Frag f;
        f.q = *reinterpret_cast<const uint4 *>(X + v * ldx + offx + 8 * piece);
        const float g = bf2f(dY[v * ldy + offy]);
#pragma unroll
        for (int e = 0; e < 8; ++e) s[e] += g * bf2f(f.h[e]);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) red[t][e] = s[e];
    __syncthreads();
    for (int w = lanes / 2; w > 0; w >>= 1) {
        if (lane < w) {
#pragma unroll
            for (int e = 0; e < 8; ++e) red[t][e] += red[t + w * c8][e];
        }
        __syncthreads();
    }
    // the row of Kp weights: 8 c8 channels, the rest zero
    if (t < Kp) P[(int64_t)blockIdx.x * Kp + t] = t < 8 * c8 ? red[t / 8][t % 8] : 0.0f;
}

// the LDS-staged kernel takes 3x3x3 layers with up to 32 output channels on
// volumes of at least 16^3
constexpr int kLdsMinN = 16;
// layers of 16 to 48 input and more than 32 output channels: a plain BF16 output
// (16-byte aligned, no FP32 copy) is summed in the LDS-tile kernel's k order from
// this edge on, below it, as all their other outputs, in the GEMM-tiled kernel's
constexpr int kZmGroupOrderN = 96;

// The GEMM-tiled kernel's launch: 64 x 64 blocks, stages of 64 k, and the
// number of slices the stage range is split into when a workspace for the
// partials is given -- enough work-groups for 4 per CU, at least 4 stages
// per slice.
struct GemmPlan {
    int mblocks, nblocks, stages, slices;
};
GemmPlan gemm_plan(int n, int cin, int cout, bool split) {
    GemmPlan p;
    const int64_t nvox = (int64_t)n * n * n;
    p.mblocks = (int)((nvox + kGemmBM - 1) / kGemmBM);
    p.nblocks = (cout + kGemmBN - 1) / kGemmBN;
    p.stages = (lgdhip_conv3d_kpad(cin, 3) + kGemmBK - 1) / kGemmBK;
    p.slices = 1;
    const int64_t base = (int64_t)p.mblocks * p.nblocks, target = 4 * lgdhip::kCUs;
    if (split && base < target) {
        const int64_t want = (target + base - 1) / base;
        p.slices = (int)std::max<int64_t>(1, std::min<int64_t>(want, p.stages / 4));
    }
    return p;
}
size_t gemm_workspace_bytes(int n, const GemmPlan &p) {
    if (p.slices <= 1) return 0;
    return (size_t)p.slices * (size_t)n * n * n * (size_t)p.nblocks * kGemmBN * 4;
}
// the layers the GEMM-tiled kernel takes (16-byte input rows; the caller
// has checked ldx, offx and the alignment when cin % 8 == 0): 3x3x3 with
// cin % 8 == 0 and more than 16 output channels below 64^3, and any size
// with more than 32 (the LDS-tile kernel takes 32 channels from 64^3 on;
// 16-channel layers stay with the z-marching kernel and, for the launches it
// does not take, the LDS-tile kernel, which sums in the same k order)
bool gemm_applies(int n, int cin, int ksize, int cout) {
    return ksize == 3 && (cin & 7) == 0 && cout > 16 && (n < 64 || cout > 32);
}

// conv3d_fwd_zm's launch: output tiles per slice (as many as the weight
// fragments' registers allow), columns and z planes per chunk
struct ZmPlan {
    int nt, slices, bx, by, bz, zchunk;
    double steps;  // modelled length of the launch in plane steps
};
ZmPlan zm_plan_of(int n, int groups, int tiles, int nt) {
    ZmPlan z;
    z.nt = nt;
    const int resident = zm_waves(groups, z.nt) >= 2 ? 2 : 1;
    z.slices = tiles / z.nt;
    z.bx = (n + 15) / 16;
    z.by = (n + 7) / 8;
    // Chunks of equal length, by the plane steps of the longest work-group:
    // where two work-groups share a CU, a step of one that has the CU alone
    // takes 0.6 of a step of two (0.8 from 5 input groups on); a chunk reads
    // two planes beyond its own and starts in about one step more.
    z.steps = 1e300;
    for (int chunks = 1; chunks <= n; ++chunks) {
        const int zc = (n + chunks - 1) / chunks;
        if ((n + zc - 1) / zc != chunks) continue;
        const int64_t on_cu = ((int64_t)z.bx * z.by * z.slices * chunks + lgdhip::kCUs - 1) / lgdhip::kCUs;
        double rounds = resident == 1 ? (double)on_cu : (double)((on_cu + 1) / 2);
        if (resident == 2 && on_cu == 1) rounds = groups <= 4 ? 0.6 : 0.8;
        const double steps = rounds * (zc + 3);
        if (steps < z.steps) {
            z.steps = steps;
            z.zchunk = zc;
            z.bz = chunks;
        }
    }
    return z;
}
ZmPlan zm_plan(int n, int groups, int cout, bool masked) {
    const int tiles = cout / 16;
    int nt = std::max(1, std::min(3, 4 / groups));
    while (tiles % nt) --nt;
    const ZmPlan z = zm_plan_of(n, groups, tiles, nt);
    // a masked row's weights are loaded value by value, 56 nt of them a lane before
    // the march begins: one tile per slice where the launch gets no longer than that
    // by it (us with nt tiles / one: 16^3 3 -> 48 11.4 / 6.2, 31^3 3 -> 48 11.8 / 8.2,
    // 24^3 3 -> 32 8.9 / 7.0; 16^3 and 17^3 3 -> 48 took 9 in conv3d_fwd_mfma)
    if (masked && nt > 1) {
        const ZmPlan one = zm_plan_of(n, groups, tiles, 1);
        if (one.steps <= z.steps + 1.25 * (nt - 1)) return one;
    }
    return z;
}

// voxel tiles per wave of the forward kernel: weight-fragment reuse bounded
// by the accumulator registers (MT x NT x 4)
constexpr int fwd_mt(int nt) { return nt <= 4 ? 4 : (nt <= 8 ? 2 : 1); }

// Forward launch shape for nvox voxels and nt cout tiles: NT tiles per wave
// (a divisor of nt), MT voxel tiles per wave (at most fwd_mt(NT)), nt / NT
// cout groups.  Takes the fewest fragment loads per MFMA (1/NT + 1/MT) among
// the shapes that give at least kFwdWaves waves (8 per CU: the 16^3 and 32^3
// levels of the U-Net otherwise leave most CUs idle), else the most waves.
constexpr int64_t kFwdWaves = 2048;
struct FwdShape {
    int nt, mt, groups;
};
FwdShape fwd_shape(int64_t nvox, int nt) {
    FwdShape best{nt, fwd_mt(nt), 1}, most = best;
    double best_loads = 1e30;
    int64_t most_waves = -1;
    for (int ntw = nt; ntw >= 1; --ntw) {
        if (nt % ntw) continue;
        for (int mt = fwd_mt(ntw); mt >= 1; mt /= 2) {
            const int64_t waves = (nvox + 16 * mt - 1) / (16 * mt) * (nt / ntw);
            const double loads = 1.0 / ntw + 1.0 / mt;
            if (waves >= kFwdWaves && loads < best_loads) {
                best_loads = loads;
                best = FwdShape{ntw, mt, nt / ntw};
            }
            if (waves > most_waves) {
                most_waves = waves;
                most = FwdShape{ntw, mt, nt / ntw};
            }
        }
    }
    return best_loads < 1e30 ? best : most;
}

// dW partial over a chunk of voxels: P[chunk][co][k] = sum_v dY[v][co] X[v+tap(k)][ci(k)]
// one wave per (chunk, k tile of 16), all co tiles; work-groups in XCD
// order (XCD c takes the contiguous range [c per, (c + 1) per): a chunk's
// waves and its neighbours share one L2)
template <int NT>
__global__ __launch_bounds__(256) void conv3d_wgrad_mfma(const u16 *__restrict__ X, int n, int ldx, int offx, int cin,
                                                         int ksize, const u16 *__restrict__ dY, int ldy, int offy,
                                                         int cout, int Kp, int chunk_vox, float *__restrict__ P,
                                                         unsigned per) {
    const int lane = threadIdx.x & 63;
    const int ktiles = Kp / 16;
    const int wave = (int)(lgdhip::xcd_tile(blockIdx.x, per, true) * 4 + threadIdx.x / 64);
    const int nvox = n * n * n;
    const int chunks = (nvox + chunk_vox - 1) / chunk_vox;
    if (wave >= chunks * ktiles) return;
    const int kt = wave % ktiles;
    const int chunk = wave / ktiles;
    const int i = lane & 15;
    const int vq = lane >> 4;
    const int K = (ksize == 1 ? 1 : 27) * cin;
    const int k = kt * 16 + i;  // this lane's B column
    int tap = 0, ci = 0, dz = 0, dy = 0, dx = 0;
    if (k < K) {
        tap = k / cin;
        ci = k % cin;
        tap_offset(tap, ksize, dz, dy, dx);
    }
    f32x4 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int v_begin = chunk * chunk_vox;
    const int v_end = min(v_begin + chunk_vox, nvox);
    // coordinates of this lane group's first voxel vb + 8 vq, carried along
    // (one voxel per element, 32 per iteration) instead of divided out per
    // element
    int x0 = (v_begin + 8 * vq) % n, y0 = ((v_begin + 8 * vq) / n) % n, z0 = (v_begin + 8 * vq) / (n * n);
    auto advance = [n](int &xa, int &ya, int &za, int by) {
        xa += by;
        while (xa >= n) {
            xa -= n;
            if (++ya == n) {
                ya = 0;
                ++za;
            }
        }
    };
    for (int vb = v_begin; vb < v_end; vb += 32) {
        Frag b;
        int x = x0, y = y0, z = z0;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int v = vb + 8 * vq + e;
            u16 val = 0;
            if (v < v_end && k < K) {
                const int zz = z + dz, yy = y + dy, xx = x + dx;
                if ((unsigned)zz < (unsigned)n && (unsigned)yy < (unsigned)n && (unsigned)xx < (unsigned)n)
                    val = X[((int64_t)((zz * n + yy) * n + xx)) * ldx + offx + ci];
            }
            b.h[e] = val;
            if (++x == n) {  // the next voxel
                x = 0;
                if (++y == n) {
                    y = 0;
                    ++z;
                }
            }
        }
        advance(x0, y0, z0, 32);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            Frag a;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int v = vb + 8 * vq + e;
                const int co = t * 16 + i;
                a.h[e] = (v < v_end && co < cout) ? dY[(int64_t)v * ldy + offy + co] : (u16)0;
            }
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, b.v, acc[t], 0, 0, 0);
        }
    }
    // D[co][k]: lane c + 16*(r/4) holds row 4*(lane/16)+e (co), column lane%16 (k)
#pragma unroll
    for (int t = 0; t < NT; ++t) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int co = t * 16 + 4 * vq + e;
            if (co < cout) P[((int64_t)chunk * cout + co) * Kp + kt * 16 + i] = acc[t][e];
        }
    }
}

// dW partials of a 3x3x3 layer straight from the channels-last tensors:
// P[chunk][co][tap*cin + ci] = sum over the chunk's voxels v of dY[v][co] X[v + tap][ci].
// A work-group owns a 16 x 8 column of voxels and marches a chunk of z planes;
// TI ci tiles and TO co tiles of 16 channels pass through LDS as one X plane
// (18 x 10 voxels with halo) and one dY plane per step, double buffered.  The
// products sum over voxels, so both MFMA operands need 8 voxels of one channel
// per lane: ds_read_b64_tr_b16 transposes 4 voxels x 16 channels while reading
// them, so no transposed copy of the tensors is made.  Wave (ti, to, ks) takes
// one pair of channel tiles and every KS-th of the plane's four 32-voxel steps
// (two 16-voxel rows): per step and X plane z it reads 9 X fragments (the dy, dx
// taps) and one new dY fragment, that of plane z + 1; with the kept ones of
// planes z and z - 1 they make all 27 taps' products (an X plane serves dz = -1,
// 0, 1 for the dY planes z + 1, z, z - 1).  108 accumulator registers per wave;
// the KS waves of a tile pair are summed through LDS in a fixed order.
//
// Per MFMA (16 cycles) the wave reads 10/27 of a fragment (8 LDS cycles), so the
// matrix cores, not LDS, bound the loop; at 16 channels the launch is bound by
// its one pass over memory.  MI355X, reduction included: 128^3 16 -> 16 42 us
// (voxel-blocked copies and a kernel reading them: 207), 48 -> 16 104 us (570),
// 64^3 96 -> 32 59 us (154); with one plane in flight instead of two 73 + 6 us
// and 106 + 12 us at 128^3.  Volumes of n % 8 != 0 had the gather kernel only
// (60^3 32 -> 32: 30 us, 250 before).
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef s16x4 __attribute__((address_space(3))) *ls_ptr;
constexpr int kWgX = 18, kWgVox = 18 * 10, kWgOut = 16 * 8;

template <int TI, int TO, int KS, int IN>
__global__ __launch_bounds__(64 * TI * TO * KS, TI * TO * KS == 4 ? 3 : 1) void conv3d_wgrad_zm(const u16 *__restrict__ X, int n, int ldx,
                                                                     int offx, int cin, const u16 *__restrict__ dY,
                                                                     int ldy, int offy, int cout, int Kp, int zchunk,
                                                                     int bx, int by, int gi, int go,
                                                                     float *__restrict__ P, unsigned groups,
                                                                     unsigned per) {
    constexpr int T = 64 * TI * TO * KS;
    constexpr int PX = kWgVox * 2 * TI, PY = kWgOut * 2 * TO;  // 16-byte pieces of a plane
    constexpr int PERX = (PX + T - 1) / T, PERY = (PY + T - 1) / T;
    constexpr int NKS = 4 / KS;                                // 32-voxel steps per wave and plane
    constexpr int kStage = 2 * (PX + PY);                      // uint4: [X buffers][dY buffers]
    constexpr int kRed = KS > 1 ? KS / 2 * TI * TO * 9 * 64 : 0;  // uint4 (4 floats): a dz's accumulators of half the waves
    __shared__ uint4 smem[kStage > kRed ? kStage : kRed];
    __shared__ int overflow;
    uint4 *const xs = smem, *const ys = smem + 2 * PX;
    unsigned b = lgdhip::xcd_tile(blockIdx.x, per, true);
    if (b >= groups) return;  // whole work-group, before any barrier
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ks = wave % KS, ti = wave / KS % TI, to = wave / KS / TI;
    const int x0 = (int)(b % bx) * 16;
    b /= bx;
    const int y0 = (int)(b % by) * 8;
    b /= by;
    const int ig = (int)(b % gi);
    b /= gi;
    const int og = (int)(b % go);
    const int zc = (int)(b / go);
    const int zs = zc * zchunk, ze = min(zs + zchunk, n);
    const int ci0 = ig * TI * 16, co0 = og * TO * 16;

    // staging: piece k is half g % 2 of tile g / 2 of voxel k / (2 T.): consecutive
    // threads read consecutive 16 bytes of a voxel's channels
    const gh_ptr zero = (gh_ptr)(const void *)kZero16;
    const gh_ptr xg = (gh_ptr)X + offx, yg = (gh_ptr)dY + offy;
    int xofs[PERX], yofs[PERY];
    bool xok[PERX], yok[PERY];
#pragma unroll
    for (int p = 0; p < PERX; ++p) {
        const int k = tid + T * p, v = k / (2 * TI), c = ci0 + 8 * (k % (2 * TI));
        const int xx = x0 + v % kWgX - 1, yy = y0 + v / kWgX - 1;
        xok[p] = k < PX && c < cin && (unsigned)xx < (unsigned)n && (unsigned)yy < (unsigned)n;
        xofs[p] = xok[p] ? (yy * n + xx) * ldx + c : 0;
    }
#pragma unroll
    for (int p = 0; p < PERY; ++p) {
        const int k = tid + T * p, v = k / (2 * TO), c = co0 + 8 * (k % (2 * TO));
        const int xx = x0 + v % 16, yy = y0 + v / 16;
        yok[p] = k < PY && c < cout && xx < n && yy < n;
        yofs[p] = yok[p] ? (yy * n + xx) * ldy + c : 0;
    }
    uint4 sx[2][PERX], sy[2][PERY];  // two planes in flight
    auto load_x = [&](int set, int z) {
        const bool ok = (unsigned)z < (unsigned)n;
        const gh_ptr base = xg + (int64_t)(ok ? z : 0) * n * n * ldx;
#pragma unroll
        for (int p = 0; p < PERX; ++p) {
            Frag f;
            f.q = load_global16(ok && xok[p] ? base + xofs[p] : zero);
            if (IN == kInMasked) {
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (e >= cin) f.h[e] = 0;
            }
            sx[set][p] = f.q;
        }
    };
    auto load_y = [&](int set, int z) {  // planes outside the chunk hold zeros
        const bool ok = z >= zs && z < ze;
        const gh_ptr base = yg + (int64_t)(ok ? z : 0) * n * n * ldy;
#pragma unroll
        for (int p = 0; p < PERY; ++p) sy[set][p] = load_global16(ok && yok[p] ? base + yofs[p] : zero);
    };
    auto store_xy = [&](int set, int buf) {
#pragma unroll
        for (int p = 0; p < PERX; ++p) {
            const int k = tid + T * p, v = k / (2 * TI), g = k % (2 * TI);
            if (k < PX) xs[buf * PX + ((g >> 1) * kWgVox + v) * 2 + (g & 1)] = sx[set][p];
        }
#pragma unroll
        for (int p = 0; p < PERY; ++p) {
            const int k = tid + T * p, v = k / (2 * TO), g = k % (2 * TO);
            if (k < PY) ys[buf * PY + ((g >> 1) * kWgOut + v) * 2 + (g & 1)] = sy[set][p];
        }
    };
    // a fragment's 8 voxels: lane group q = lane / 16 takes x 4 (q & 1) .. + 3 and
    // 8 further of row q / 2 of the step's two, the same for X and dY; lane t of
    // the group addresses voxel t / 4, channels 4 (t % 4) .. + 3
    const int q = lane >> 4, t = lane & 15;
    const int xv = 4 * (q & 1) + (t >> 2), row = q >> 1;
    typedef const char __attribute__((address_space(3))) *lc_ptr;
    const lc_ptr xlane = (lc_ptr)(void *)xs + (ti * kWgVox + row * kWgX + xv) * 32 + (t & 3) * 8;
    const lc_ptr ylane = (lc_ptr)(void *)ys + (to * kWgOut + row * 16 + xv) * 32 + (t & 3) * 8;
    auto frag = [](lc_ptr p) {
        union {
            s16x4 s[2];
            Frag f;
        } u;
        u.s[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ls_ptr)p);
        u.s[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ls_ptr)(p + 8 * 32));
        return u.f;
    };

    f32x4 acc[3][9];
    Frag a[3][NKS];  // dY of planes z + 1, z, z - 1
    auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
#pragma unroll
            for (int e = 0; e < 9; ++e) acc[d][e] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < NKS; ++s) a[d][s].q = make_uint4(0u, 0u, 0u, 0u);
        }
    };
    // the products of X plane z, in buffer PH with dY plane z + 1
    auto products = [&](auto ph_c, auto masked_c, int z) __attribute__((always_inline)) {
        constexpr int PH = decltype(ph_c)::value;
        constexpr bool MASKED = decltype(masked_c)::value;
#pragma unroll
        for (int s = 0; s < NKS; ++s) {
            const int step = ks + KS * s;  // rows 2 step, 2 step + 1
            a[2][s] = a[1][s];
            a[1][s] = a[0][s];
            a[0][s] = frag(ylane + PH * PY * 16 + step * 2 * 16 * 32);
            const lc_ptr xp = xlane + PH * PX * 16 + step * 2 * kWgX * 32;
            uint32_t in[4];  // MASKED: the fragment's voxels whose dY is inside the volume
            if (MASKED) {
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const int xx = x0 + 4 * (q & 1) + 8 * (w / 2) + 2 * (w % 2);
                    const bool yin = y0 + 2 * step + row < n;
                    in[w] = (yin && xx < n ? 0xFFFFu : 0u) | (yin && xx + 1 < n ? 0xFFFF0000u : 0u);
                }
            }
#pragma unroll
            for (int e = 0; e < 9; ++e) {  // tap (dy, dx) = (e / 3 - 1, e % 3 - 1)
                const Frag f = frag(xp + ((e / 3) * kWgX + e % 3) * 32);
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    Frag g = f;
                    if (MASKED) {
                        const uint32_t zin = z + 1 - d >= zs && z + 1 - d < ze ? ~0u : 0u;
                        g.q = make_uint4(f.q.x & in[0] & zin, f.q.y & in[1] & zin, f.q.z & in[2] & zin,
                                         f.q.w & in[3] & zin);
                    }
                    acc[d][e] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[d][s].v, g.v, acc[d][e], 0, 0, 0);
                }
            }
        }
    };

    if (tid == 0) overflow = 0;
    clear();
    load_x(0, zs - 1);
    load_y(0, zs);
    load_x(1, zs);
    load_y(1, zs + 1);
    store_xy(0, 0);
    __syncthreads();
    // step at X plane z (dY plane z + 1) in buffer PH: the planes of step z + 2 go
    // out, those of z + 1 (in flight for a whole step) are stored after the products;
    // LAST: z may be (1) or is (2) the last plane, after which nothing is stored
    auto plane = [&](auto ph_c, auto last_c, int z) __attribute__((always_inline)) {
        constexpr int PH = decltype(ph_c)::value, LAST = decltype(last_c)::value;
        load_x(PH, z + 2);
        load_y(PH, z + 3);
        products(ph_c, lgdhip::ic<0>{}, z);
        if (LAST == 0 || (LAST == 1 && z < ze)) {
            store_xy(PH ^ 1, PH ^ 1);
            __syncthreads();
        }
    };
    int z = zs - 1;
    for (; z + 1 <= ze; z += 2) {
        plane(lgdhip::ic<0>{}, lgdhip::ic<0>{}, z);
        plane(lgdhip::ic<1>{}, lgdhip::ic<1>{}, z + 1);
    }
    if (z <= ze) plane(lgdhip::ic<0>{}, lgdhip::ic<2>{}, z);
    // Voxels outside the chunk or the volume add dY = 0 times a real X, which is
    // NaN where that X is infinite.  If a sum is not finite, the chunk is summed
    // again without those X, one plane at a time; on finite tensors the test costs
    // up to 1.4 us a launch (128^3 16 -> 16 40.9 us without, 41.5 with, 64^3 32 ->
    // 32 26.5 and 27.9).  Masks in the march itself spilled 20 to 290 registers.
    f32x4 sum = acc[0][0];
#pragma unroll
    for (int k = 1; k < 27; ++k) sum += acc[k / 9][k % 9];
    const float all = sum[0] + sum[1] + sum[2] + sum[3];
    if (!(fabsf(all) < INFINITY)) overflow = 1;
    __syncthreads();
    if (__builtin_expect(overflow != 0, 0)) {
        clear();
        for (z = zs - 1; z <= ze; ++z) {
            load_x(0, z);
            load_y(0, z + 1);
            store_xy(0, 0);
            __syncthreads();
            products(lgdhip::ic<0>{}, lgdhip::ic<1>{}, z);
            __syncthreads();
        }
    }
    // sum the KS waves of each tile pair, one dz at a time: the upper half of the
    // waves writes, the lower half adds
    if (KS > 1) {
        f32x4 *red = reinterpret_cast<f32x4 *>(smem);
        const int pair = to * TI + ti;
#pragma unroll
        for (int d = 0; d < 3; ++d)
#pragma unroll
            for (int half = KS / 2; half >= 1; half /= 2) {
                if (ks >= half && ks < 2 * half) {
#pragma unroll
                    for (int e = 0; e < 9; ++e) red[((pair * (KS / 2) + ks - half) * 9 + e) * 64 + lane] = acc[d][e];
                }
                __syncthreads();
                if (ks < half) {
#pragma unroll
                    for (int e = 0; e < 9; ++e) acc[d][e] += red[((pair * (KS / 2) + ks) * 9 + e) * 64 + lane];
                }
                __syncthreads();
            }
        if (ks != 0) return;
    }
    // D lane layout: row (co) 4 (lane / 16) + e, column (ci) lane % 16
    const int64_t chunk = ((int64_t)zc * by + y0 / 8) * bx + x0 / 16;
    const int ci = ci0 + ti * 16 + t;
    if (ci >= cin) return;
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int k = 0; k < 9; ++k)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int co = co0 + to * 16 + 4 * q + e;
                if (co < cout) P[(chunk * cout + co) * Kp + (9 * d + k) * cin + ci] = acc[d][k][e];
            }
}

// dW[co][k] = sum over chunks of P (fixed order) for k < K; the padding
// columns k >= K stay zero
// A work-group of 64 x ROWS threads takes 64 consecutive outputs; thread row j
// sums the chunks j, j + ROWS, j + 2 ROWS, ... (eight loads in flight, coalesced
// across the 64 outputs) and the row sums are added in row order: a fixed
// order for every output.  16 rows where the outputs are fewer than two
// work-groups per CU and have more than 16 chunks (16 -> 16: 112 of them; 128^3 40.1 us with the column kernel,
// 44.1 with 4 rows), else 4: wide layers have few chunks on small volumes, and
// rows without one cost their launch (16^3 128 -> 128 21.3 us, 32.0 with 16 rows).
// The same holds for 16 chunks or fewer: 1^3 7.9 us with 4 rows, 9.6 with 16, 4^3
// 9.2 / 10.3, 8^3 11.2 / 11.8 (mean over 48 layers; alike with 16 to 64 chunks).
constexpr int kWgradReduceOutputs = 64;
template <int ROWS>
__global__ __launch_bounds__(kWgradReduceOutputs *ROWS) void conv3d_wgrad_reduce(const float *__restrict__ P,
                                                                                 int chunks, int cout, int Kp, int K,
                                                                                 float *__restrict__ dW,
                                                                                 int accumulate) {
    __shared__ float part[ROWS][kWgradReduceOutputs];
    const int total = cout * Kp;  // < 2^31: cout <= 192, Kp <= 27 * 192 + 31
    const int o = (int)blockIdx.x * kWgradReduceOutputs + (int)threadIdx.x;
    const int j = (int)threadIdx.y;
    float s = 0.0f;
    if (o < total && o % Kp < K) {
#pragma unroll 8
        for (int c = j; c < chunks; c += ROWS) s += P[(int64_t)c * total + o];
    }
    part[j][threadIdx.x] = s;
    __syncthreads();
    if (j != 0 || o >= total) return;
    float r = part[0][threadIdx.x];
#pragma unroll
    for (int k = 1; k < ROWS; ++k) r += part[k][threadIdx.x];
    if (o % Kp >= K) {  // padding columns stay zero
        dW[o] = accumulate ? dW[o] : 0.0f;
        return;
    }
    dW[o] = accumulate ? dW[o] + r : r;
}

// db: channel sums over chunks of 8192 voxels, then a fixed-order sum of the
// chunks
constexpr int kBiasChunk = 8192;
__global__ void row_sum_final(const float *__restrict__ Pb, int bchunks, int cout, float *__restrict__ db,
                              int accumulate) {
    const int co = blockIdx.x * blockDim.x + threadIdx.x;
    if (co >= cout) return;
    float s = 0.0f;
    for (int c = 0; c < bchunks; ++c) s += Pb[co * bchunks + c];
    db[co] = accumulate ? db[co] + s : s;
}

// db[co] partial sums over chunks of 8192 voxels, channels-last rows of any
// stride: thread t of a block handles channel t % cout of every (256 / cout)-th
// voxel, so a wave reads whole voxel rows (coalesced); fixed-order sums
__global__ __launch_bounds__(256) void bias_grad_partial(const u16 *__restrict__ dY, int64_t nvox, int ldy, int offy,
                                                         int cout, float *__restrict__ Pb, int bchunks) {
    __shared__ float red[256];
    const int c = blockIdx.x;
    const int lanes = 256 / cout;  // voxel lanes
    const int t = threadIdx.x;
    float s = 0.0f;
    if (t < lanes * cout) {
        const int co = t % cout, vl = t / cout;
        const int64_t v0 = (int64_t)c * kBiasChunk;
        const int64_t v1 = v0 + kBiasChunk < nvox ? v0 + kBiasChunk : nvox;
        for (int64_t v = v0 + vl; v < v1; v += lanes) s += bf2f(dY[v * ldy + offy + co]);
    }
    red[t] = s;
    __syncthreads();
    if (t < cout) {
        float sum = 0.0f;
        for (int vl = 0; vl < lanes; ++vl) sum += red[vl * cout + t];
        Pb[t * bchunks + c] = sum;
    }
}

// db[co] partial sums over chunks of 8192 voxels of aligned rows of whole
// 8-channel pieces: a work-group takes NP pieces of one chunk, thread t the
// voxels t, t + 256, .. of the chunk (at most 32, all loads independent), and
// the 256 sums of a channel are added as a tree.  Bound by latency on small
// volumes, by its pass over dY on large ones.  bias_grad_partial, which takes the
// other rows, has one work-group per chunk and 256 / cout voxel lanes, chains of
// up to 8192 additions and one busy CU for a 16^3 layer.  What db adds to a
// weight gradient (us, here / there): 128^3 x 16 29 / 138, 64^3 x 32 13 / 253,
// 32^3 x 64 13 / 494, 16^3 x 128 8 / 198; a training step with biases at 128^3
// takes 2263 us against 6846.
template <int NP>
__global__ __launch_bounds__(256) void bias_grad_rows(const u16 *__restrict__ dY, int64_t nvox, int ldy, int offy,
                                                      float *__restrict__ Pb, int bchunks) {
    constexpr int CH = 8 * NP;
    __shared__ float red[CH][256];
    const int t = threadIdx.x, c = blockIdx.x, co = (int)blockIdx.y * CH;
    const int64_t v0 = (int64_t)c * kBiasChunk;
    const int64_t v1 = v0 + kBiasChunk < nvox ? v0 + kBiasChunk : nvox;
    float s[CH] = {};
#pragma unroll 4
    for (int64_t v = v0 + t; v < v1; v += 256) {
        Frag f[NP];
#pragma unroll
        for (int p = 0; p < NP; ++p) f[p].q = *reinterpret_cast<const uint4 *>(dY + v * ldy + offy + co + 8 * p);
#pragma unroll
        for (int k = 0; k < CH; ++k) s[k] += bf2f(f[k / 8].h[k % 8]);
    }
#pragma unroll
    for (int k = 0; k < CH; ++k) red[k][t] = s[k];
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        for (int i = t; i < CH * w; i += 256) red[i / w][i % w] += red[i / w][i % w + w];
        __syncthreads();
    }
    if (t < CH) Pb[(co + t) * bchunks + c] = red[t][0];
}

// dgrad weights: Wt[ci][tap'*cout + co] = W[co][tap*cin + ci], tap' = 26 - tap
__global__ void conv3d_dgrad_weights(const u16 *__restrict__ W, int cin, int cout, int ksize, int Kp,
                                     u16 *__restrict__ Wt, int Kpt) {
    const int taps = ksize == 1 ? 1 : 27;
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (int64_t)cin * Kpt) return;
    const int ci = (int)(idx / Kpt);
    const int kk = (int)(idx % Kpt);
    u16 v = 0;
    if (kk < taps * cout) {
        const int tp = kk / cout, co = kk % cout;
        const int tap = taps - 1 - tp;
        v = W[(int64_t)co * Kp + tap * cin + ci];
    }
    Wt[idx] = v;
}

// g *= (y > 0) for the ReLU backward (in place, BF16)
__global__ void relu_backward(u16 *g, int ldg, int offg, const u16 *__restrict__ y, int ldy, int offy, int c,
                              int64_t nvox) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= nvox * c) return;
    const int64_t v = idx / c;
    const int ch = (int)(idx % c);
    if (!(bf2f(y[v * ldy + offy + ch]) > 0.0f)) g[v * ldg + offg + ch] = 0;
}

// 2x2x2 average pool: Y (n/2)^3 <- X n^3
__global__ void avgpool2(const u16 *__restrict__ X, int n, int ldx, int offx, u16 *Y, int ldy, int offy, int c) {
    const int m = n / 2;
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (int64_t)m * m * m * c) return;
    const int ch = (int)(idx % c);
    const int64_t v = idx / c;
    const int x = (int)(v % m), y = (int)((v / m) % m), z = (int)(v / ((int64_t)m * m));
    float s = 0.0f;
    for (int d = 0; d < 8; ++d) {
        const int zz = 2 * z + (d >> 2), yy = 2 * y + ((d >> 1) & 1), xx = 2 * x + (d & 1);
        s += bf2f(X[((int64_t)((zz * n + yy) * n + xx)) * ldx + offx + ch]);
    }
    Y[v * ldy + offy + ch] = f2bf(s * 0.125f);
}

// gradient of the average pool: dX[child] (+)= dY[parent] / 8
__global__ void avgpool2_backward(const u16 *__restrict__ dY, int n, int ldy, int offy, u16 *dX, int ldx, int offx,
                                  int c, int accumulate) {
    const int m = n / 2;
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (int64_t)n * n * n * c) return;
    const int ch = (int)(idx % c);
    const int64_t v = idx / c;
    const int x = (int)(v % n), y = (int)((v / n) % n), z = (int)(v / ((int64_t)n * n));
    const int64_t p = ((int64_t)(z / 2) * m + y / 2) * m + x / 2;
    float g = bf2f(dY[p * ldy + offy + ch]) * 0.125f;
    u16 *q = dX + v * ldx + offx + ch;
    if (accumulate) g += bf2f(*q);
    *q = f2bf(g);
}

// nearest 2x upsample: Y (2m)^3 <- X m^3
__global__ void upsample2(const u16 *__restrict__ X, int m, int ldx, int offx, u16 *Y, int ldy, int offy, int c) {
    const int n = 2 * m;
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (int64_t)n * n * n * c) return;
    const int ch = (int)(idx % c);
    const int64_t v = idx / c;
    const int x = (int)(v % n), y = (int)((v / n) % n), z = (int)(v / ((int64_t)n * n));
    const int64_t p = ((int64_t)(z / 2) * m + y / 2) * m + x / 2;
    Y[v * ldy + offy + ch] = X[p * ldx + offx + ch];
}

// gradient of the upsample: dX[parent] = sum of the 8 children
__global__ void upsample2_backward(const u16 *__restrict__ dY, int m, int ldy, int offy, u16 *dX, int ldx, int offx,
                                   int c, int accumulate) {
    const int n = 2 * m;
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (int64_t)m * m * m * c) return;
    const int ch = (int)(idx % c);
    const int64_t v = idx / c;
    const int x = (int)(v % m), y = (int)((v / m) % m), z = (int)(v / ((int64_t)m * m));
    float s = 0.0f;
    for (int d = 0; d < 8; ++d) {
        const int zz = 2 * z + (d >> 2), yy = 2 * y + ((d >> 1) & 1), xx = 2 * x + (d & 1);
        s += bf2f(dY[((int64_t)((zz * n + yy) * n + xx)) * ldy + offy + ch]);
    }
    u16 *q = dX + v * ldx + offx + ch;
    if (accumulate) s += bf2f(*q);
    *q = f2bf(s);
}

// The same four resampling kernels over 8 channels per thread (16-byte loads
// and stores), used when the channel count, row strides, channel offsets and
// base pointers are multiples of 8 elements.  Each channel is summed in the
// order of the kernels above, so the results are bit-identical.
struct alignas(16) Bf8 {
    u16 h[8];
};
__device__ __forceinline__ Bf8 ld8(const u16 *p) { return *reinterpret_cast<const Bf8 *>(p); }
__device__ __forceinline__ void st8(u16 *p, const Bf8 &v) { *reinterpret_cast<Bf8 *>(p) = v; }

// g *= (y > 0), 8 channels per thread; items = voxels * c8 < 2^31.  Dense
// tensors (c8 0: both strides the channel count) need no division.  At 128^3 x
// 16 channels one element per thread with a 64-bit division took 74 us.
__global__ void relu_backward_v8(u16 *__restrict__ g, int ldg, int offg, const u16 *__restrict__ y, int ldy, int offy,
                                 int c8, uint32_t items) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= items) return;
    int64_t ig = (int64_t)i * 8, iy = ig;
    if (c8 > 0) {
        const uint32_t v = i / (uint32_t)c8, ch = 8 * (i - v * (uint32_t)c8);
        ig = (int64_t)v * ldg + offg + ch;
        iy = (int64_t)v * ldy + offy + ch;
    }
    const Bf8 a = ld8(y + iy);
    Bf8 o = ld8(g + ig);
#pragma unroll
    for (int k = 0; k < 8; ++k)
        if (!(bf2f(a.h[k]) > 0.0f)) o.h[k] = 0;
    st8(g + ig, o);
}

// Thread coordinates of the 8-channel resampling kernels over a w^3 volume:
// a launch row_grid(w, c8) gives each (y, z) row blockIdx.y / .z, and the
// threads along x cover its (x, channel chunk) pairs, the chunk fastest
// (consecutive threads, consecutive 16-byte pieces of a voxel's channels).
// 32-bit arithmetic throughout (a flat 64-bit index divided by run-time
// extents costs hundreds of instructions per thread).
__device__ __forceinline__ bool row_thread(int w, int c8, int &x, int &ch) {
    const int t = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (t >= w * c8) return false;
    x = t / c8;
    ch = (t - x * c8) * 8;
    return true;
}

__global__ void avgpool2_v8(const u16 *__restrict__ X, int n, int ldx, int offx, u16 *Y, int ldy, int offy, int c8) {
    const int m = n / 2;
    int x, ch;
    if (!row_thread(m, c8, x, ch)) return;
    const int y = blockIdx.y, z = blockIdx.z;
    const int64_t v = ((int64_t)z * m + y) * m + x;
    float s[8] = {};
    for (int d = 0; d < 8; ++d) {
        const int zz = 2 * z + (d >> 2), yy = 2 * y + ((d >> 1) & 1), xx = 2 * x + (d & 1);
        const Bf8 a = ld8(X + ((int64_t)((zz * n + yy) * n + xx)) * ldx + offx + ch);
#pragma unroll
        for (int k = 0; k < 8; ++k) s[k] += bf2f(a.h[k]);
    }
    Bf8 o;
#pragma unroll
    for (int k = 0; k < 8; ++k) o.h[k] = f2bf(s[k] * 0.125f);
    st8(Y + v * ldy + offy + ch, o);
}

__global__ void avgpool2_backward_v8(const u16 *__restrict__ dY, int n, int ldy, int offy, u16 *dX, int ldx, int offx,
                                     int c8, int accumulate, const u16 *__restrict__ A, int lda, int offa) {
    const int m = n / 2;
    int x, ch;
    if (!row_thread(n, c8, x, ch)) return;
    const int y = blockIdx.y, z = blockIdx.z;
    const int64_t v = ((int64_t)z * n + y) * n + x;
    const int64_t p = ((int64_t)(z / 2) * m + y / 2) * m + x / 2;
    const Bf8 a = ld8(dY + p * ldy + offy + ch);
    u16 *q = dX + v * ldx + offx + ch;
    Bf8 old;
    if (accumulate) old = ld8(q);
    Bf8 o;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        float g = bf2f(a.h[k]) * 0.125f;
        if (accumulate) g += bf2f(old.h[k]);
        o.h[k] = f2bf(g);
    }
    if (A) {  // ReLU backward of the layer that made X
        const Bf8 act = ld8(A + v * lda + offa + ch);
#pragma unroll
        for (int k = 0; k < 8; ++k)
            if (!(bf2f(act.h[k]) > 0.0f)) o.h[k] = 0;
    }
    st8(q, o);
}

__global__ void upsample2_v8(const u16 *__restrict__ X, int m, int ldx, int offx, u16 *Y, int ldy, int offy, int c8) {
    const int n = 2 * m;
    int x, ch;
    if (!row_thread(n, c8, x, ch)) return;
    const int y = blockIdx.y, z = blockIdx.z;
    const int64_t v = ((int64_t)z * n + y) * n + x;
    const int64_t p = ((int64_t)(z / 2) * m + y / 2) * m + x / 2;
    st8(Y + v * ldy + offy + ch, ld8(X + p * ldx + offx + ch));
}

// Nearest 2x upsampling of x (m^3, cu channels) written together with a
// skip tensor (n^3 = (2m)^3, cs channels) as whole concatenation rows:
//   y[v][offy + c] = c < cu ? x[parent(v)][offx + c] : s[v][offs + c - cu]
// so every 128-byte line of y is written by one launch in full (the
// encoder writing its channels into the rows and the upsampling writing the
// others leave each line partly written twice, and a partial line costs
// the memory a read-modify-write).  8 channels per thread; consecutive
// threads write consecutive 16-byte pieces of a row.
__global__ void upsample2_concat_v8(const u16 *__restrict__ X, int m, int ldx, int offx, int cu8,
                                    const u16 *__restrict__ S, int lds, int offs, u16 *Y, int ldy, int offy, int c8) {
    const int n = 2 * m;
    int x, ch;
    if (!row_thread(n, c8, x, ch)) return;
    const int y = blockIdx.y, z = blockIdx.z;
    const int64_t v = ((int64_t)z * n + y) * n + x;
    Bf8 val;
    if (ch < 8 * cu8) {
        const int64_t p = ((int64_t)(z / 2) * m + y / 2) * m + x / 2;
        val = ld8(X + p * ldx + offx + ch);
    } else {
        val = ld8(S + v * lds + offs + ch - 8 * cu8);
    }
    st8(Y + v * ldy + offy + ch, val);
}

// the same, one element per thread (any channel counts, strides, offsets)
__global__ void upsample2_concat(const u16 *__restrict__ X, int m, int ldx, int offx, int cu,
                                 const u16 *__restrict__ S, int lds, int offs, int cs, u16 *Y, int ldy, int offy) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int c = cu + cs, n = 2 * m;
    if (idx >= (int64_t)n * n * n * c) return;
    const int ch = (int)(idx % c);
    const int64_t v = idx / c;
    const int x = (int)(v % n), y = (int)((v / n) % n), z = (int)(v / ((int64_t)n * n));
    u16 val;
    if (ch < cu) {
        const int64_t p = ((int64_t)(z / 2) * m + y / 2) * m + x / 2;
        val = X[p * ldx + offx + ch];
    } else {
        val = S[v * lds + offs + ch - cu];
    }
    Y[v * ldy + offy + ch] = val;
}

__global__ void upsample2_backward_v8(const u16 *__restrict__ dY, int m, int ldy, int offy, u16 *dX, int ldx, int offx,
                                      int c8, int accumulate, const u16 *__restrict__ A, int lda, int offa) {
    const int n = 2 * m;
    int x, ch;
    if (!row_thread(m, c8, x, ch)) return;
    const int y = blockIdx.y, z = blockIdx.z;
    const int64_t v = ((int64_t)z * m + y) * m + x;
    float s[8] = {};
    for (int d = 0; d < 8; ++d) {
        const int zz = 2 * z + (d >> 2), yy = 2 * y + ((d >> 1) & 1), xx = 2 * x + (d & 1);
        const Bf8 a = ld8(dY + ((int64_t)((zz * n + yy) * n + xx)) * ldy + offy + ch);
#pragma unroll
        for (int k = 0; k < 8; ++k) s[k] += bf2f(a.h[k]);
    }
    u16 *q = dX + v * ldx + offx + ch;
    Bf8 old;
    if (accumulate) old = ld8(q);
    Bf8 o;
#pragma unroll
    for (int k = 0; k < 8; ++k) o.h[k] = f2bf(accumulate ? s[k] + bf2f(old.h[k]) : s[k]);
    if (A) {  // ReLU backward of the layer that made X
        const Bf8 act = ld8(A + v * lda + offa + ch);
#pragma unroll
        for (int k = 0; k < 8; ++k)
            if (!(bf2f(act.h[k]) > 0.0f)) o.h[k] = 0;
    }
    st8(q, o);
}

// FP32 -> BF16 into a channel slot of a channels-last tensor
__global__ void pack_bf16(const float *__restrict__ src, int64_t nvox, u16 *Y, int ldy, int offy) {
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v < nvox) Y[v * ldy + offy] = f2bf(src[v]);
}

// up to 8 FP32 fields -> whole 8-channel rows, the channels past them zero (a
// fill and one pass per field, each writing 2 of every 16 bytes, took 47 us at
// 128^3 with three fields)
struct PackFields {
    const float *f[8];
};
__global__ void pack_rows_bf16(PackFields src, int count, int64_t nvox, u16 *__restrict__ Y, int ldy) {
    const int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (v >= nvox) return;
    Bf8 o;
#pragma unroll
    for (int k = 0; k < 8; ++k) o.h[k] = k < count ? f2bf(src.f[k][v]) : (u16)0;
    st8(Y + v * ldy, o);
}

// MSE loss: L = mean((pred - target)^2); grad = 2 (pred - target) / N as BF16;
// per-block partial sums of the squared error (deterministic reduction)
__global__ void mse_loss(const float *__restrict__ pred, const float *__restrict__ target, int64_t nvox, u16 *grad,
                         int ldg, float *__restrict__ partial) {
    __shared__ float lds[256];
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    float se = 0.0f;
    if (v < nvox) {
        const float d = pred[v] - target[v];
        se = d * d;
        grad[v * ldg] = f2bf(2.0f * d / (float)nvox);
    }
    lds[threadIdx.x] = se;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) lds[threadIdx.x] += lds[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = lds[0];
}

// Adam on FP32 master weights [cout][Kp] (padding columns stay zero); writes BF16 copies
__global__ void adam_step(float *__restrict__ w, float *__restrict__ m, float *__restrict__ v,
                          const float *__restrict__ g, int64_t count, int cols_used, int Kp, float lr, float b1,
                          float b2, float eps, float c1, float c2, u16 *__restrict__ wb) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    if (Kp > 0 && (int)(i % Kp) >= cols_used) {
        w[i] = 0.0f;
        if (wb) wb[i] = 0;
        return;
    }
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    w[i] = wi;
    if (wb) wb[i] = f2bf(wi);
}

unsigned blocks_for(int64_t n, int per = 256) { return (unsigned)((n + per - 1) / per); }
// the launch of a row_thread kernel over a w^3 volume with c8 chunks of 8
// channels (w <= kMaxRowGrid: the grid's y and z extents; larger volumes take
// the per-element kernels)
constexpr int64_t kMaxRowGrid = 65535;
dim3 row_grid(int w, int c8) { return dim3(blocks_for((int64_t)w * c8), (unsigned)w, (unsigned)w); }
// 8-channel (16-byte) resampling applies: channel count, strides and channel
// offsets multiples of 8 elements, both base pointers 16-byte aligned
bool vec8(const void *a, const void *b, int c, int lda, int offa, int ldb, int offb) {
    return c % 8 == 0 && lda % 8 == 0 && offa % 8 == 0 && ldb % 8 == 0 && offb % 8 == 0 &&
           ((uintptr_t)a & 15) == 0 && ((uintptr_t)b & 15) == 0;
}

// Launch of conv3d_wgrad_zm: tile pairs TI x TO and KS waves per pair, channel
// groups, z planes per chunk and chunks of the volume.
struct ZmWgrad {
    int ti, to, ks, gi, go, bx, by, zchunk, chunks;
    int64_t groups() const { return (int64_t)chunks * gi * go; }
};
constexpr struct {
    int ti, to, ks;
} kZmWgrad[] = {{1, 1, 4}, {1, 2, 4}, {2, 1, 4}, {3, 1, 4}, {2, 2, 2}, {3, 2, 1}, {2, 4, 1}, {4, 2, 1}};
// 3x3x3 layers whose 8-channel pieces are whole (or, for the network's first
// layer, one masked row); the partials index rows of channels with 32 bits
bool wgrad_zm_shape(int cin, int ksize, int cout) { return ksize == 3 && (cin % 8 == 0 || cin < 8) && cout % 8 == 0; }
// Bytes of a voxel's c channels that groups of `tiles` 16-channel tiles read among
// them when each group fetches whole 128-byte lines anew (a row below 128 bytes is
// read whole by each).
int wgrad_row_bytes(int c, int tiles) {
    int lines = 0;
    for (int a = 0; a < c; a += 16 * tiles) lines += (std::min(c, a + 16 * tiles) + 63) / 64 - a / 64;
    return lines * std::min(128, 2 * c);
}
// Bytes of a voxel's c channels that the groups fetch beyond one row: none while
// the volume stays in the L2s between the groups that share its lines; past 28 MB
// of their 32 most of each line (0.65: the least total time over 425 layers timed
// in every grouping, 2 % above the best of each; 11 % without).
double wgrad_refetch(int n, int c, int tiles) {
    const double row = 2.0 * c;
    return row * n * n * n > 28e6 ? 0.65 * std::max(0.0, wgrad_row_bytes(c, tiles) - row) : 0.0;
}
ZmWgrad wgrad_zm_plan(int n, int cin, int cout) {
    const int cit = (cin + 15) / 16, cot = (cout + 15) / 16;
    ZmWgrad best{};
    double best_us = 1e300;
    for (const auto &c : kZmWgrad) {
        if (cin < 8 && c.ti > 1) continue;  // the masked row has the one-tile kernels
        if (cin < 8 && c.to > 2) continue;
        ZmWgrad w{c.ti, c.to, c.ks, (cit + c.ti - 1) / c.ti, (cot + c.to - 1) / c.to, (n + 15) / 16, (n + 7) / 8, 0, 0};
        const int waves = c.ti * c.to * c.ks, resident = waves == 4 ? 3 : 1;
        // what the groups' shares of a 128-byte line cost on top (us): a part of the
        // grouping alone, the chunk length is chosen by the rest.  MI355X, us, without
        // it / with it: 72^3 64 -> 64 404 / 114, 72^3 64 -> 32 148 / 59, 88^3 64 -> 16
        // 120 / 71, 120^3 3 -> 128 383 / 232; it costs 108^3 3 -> 128 230 / 243.
        const double lines =
            (double)n * n * n * (w.go * wgrad_refetch(n, cin, c.ti) + w.gi * wgrad_refetch(n, cout, c.to)) / 4.5e6;
        for (int zc = 2; zc <= 64; zc *= 2) {
            w.zchunk = zc;
            w.chunks = w.bx * w.by * ((n + zc - 1) / zc);
            // Modelled time (us): a plane step of the CU's resident work-groups
            // takes its memory latency (0.7) or its products (27 MFMAs of 16
            // cycles per wave and 32-voxel step, at 0.7 of issue), a chunk two
            // halo planes and its start and reduction (4); the partials' round
            // trip at 4 TB/s and the tensors' (X with its halo) at 4.5 TB/s.
            const double on_cu = (double)((w.groups() + lgdhip::kCUs - 1) / lgdhip::kCUs);
            const double together = std::min<double>(on_cu, resident), rounds = std::ceil(on_cu / resident);
            const double products = std::max(1.0, together * waves / 4) * (4 / c.ks) * 27 * 16 / 2400.0 / 0.7;
            const double march = rounds * ((zc + 2) * std::max(0.7, products) + 4.0);
            const double partials = 2.0 * w.chunks * cout * lgdhip_conv3d_kpad(cin, 3) * 4 / 4e6;
            const double tensors = 2.0 * n * n * n * (1.4 * (zc + 2) / zc * w.go * cin + (double)w.gi * cout) / 4.5e6;
            const double us = std::max(march, tensors) + partials + lines;
            if (us < best_us) {
                best_us = us;
                best = w;
            }
        }
    }
    return best;
}

// Voxels per chunk of the general kernel when the caller leaves it to the
// library (chunk_vox <= 0): the largest power of two <= 4096 (and >= 128) that
// gives 2048 tasks.  A task is a wave's 16 columns of k, but for layers of whole
// 16-channel tiles on n % 8 == 0 up to 4 x 4 tiles (a single one with 9 taps, few
// with 3): their chunks stay 2 to 8 times shorter than 2048 waves would need, and
// the shorter serial sums are both faster and nearer to the 64-bit sums.  MI355X,
// chunks of this length / of 2048 waves, us and relative error: 64^3 16 -> 16 97,
// 2.3e-7 / 115, 3.0e-7; 64^3 32 -> 32 213, 2.4e-7 / 288, 4.2e-7; 32^3 64 -> 64 90,
// 1.5e-7 / 108, 2.2e-7; 32^3 192 -> 64 248, 2.2e-7 / 327, 4.1e-7.
int wgrad_chunk(int n, int cin, int ksize, int cout) {
    const int64_t nvox = (int64_t)n * n * n;
    int64_t tasks = lgdhip_conv3d_kpad(cin, ksize) / 16;
    if (ksize == 3 && cin % 16 == 0 && cout % 16 == 0 && n % 8 == 0) {
        const int cot = cout / 16, cit = cin / 16;
        const int ct = cot % 4 == 0 ? 4 : (cot % 2 == 0 ? 2 : 1), it = cit % 4 == 0 ? 4 : (cit % 2 == 0 ? 2 : 1);
        tasks = 27 / (ct * it <= 4 ? (ct * it == 1 ? 9 : 3) : 1) * (cot / ct) * (cit / it);
    }
    int c = 4096;
    while (c > 128 && (nvox + c - 1) / c * tasks < 2048) c /= 2;
    return c;
}

// Modelled time (us) of the general kernel on small volumes, its reduction
// included: what a wave's steps over its output tiles take, and the waves beyond
// the few that run for nothing.
double wgrad_gather_us(int n, int cin, int cout, int chunk_vox) {
    const int64_t nvox = (int64_t)n * n * n;
    const int tiles = (cout + 15) / 16;
    const double steps = (double)((std::min<int64_t>(chunk_vox, nvox) + 31) / 32);
    const double waves = (double)((nvox + chunk_vox - 1) / chunk_vox) * (lgdhip_conv3d_kpad(cin, 3) / 16);
    return 8.3 + 0.33 * tiles * steps + 0.0014 * waves * (1 + 0.2 * (tiles - 1));
}

// The column kernel takes 14 us on the smallest layers (with a masked row 0.55 more
// for each further output tile), its march and the epilogue of 27 taps.  Below that
// the general kernel is the faster one (4^3 64 -> 64 10.0 against 12.8, 12^3 32 -> 16
// 10.2 / 12.7, 16^3 3 -> 16 9.3 / 13.3, 17^3 16 -> 16 10.8 / 13.4, 16^3 24 -> 32 12.4
// / 14.3, 24^3 1 -> 64 14.4 / 16.8; over 0.75 to 1 beyond the line 13.8 on average
// against 13.9, over 1 to 1.5 15.8 / 14.5; 16^3 64 -> 64 28 / 18).
// A single input channel is 27 columns of k, two tiles for the general kernel, and a
// masked row with 27 taps for the column kernel.  With 4 output tiles or more the
// latter's groups re-fetch dY's lines on middle volumes, whose columns also leave
// many of its waves short (us, general / column: 68^3 1 -> 64 46 / 49, 88^3 1 -> 64
// 77 / 80, 68^3 1 -> 128 62 / 74, 88^3 1 -> 128 107 / 134; 64^3 1 -> 128 52 / 39,
// 96^3 1 -> 128 146 / 135).
bool wgrad_columns_pay(int n, int cin, int cout, int chunk_vox) {
    if (cin == 1 && cout > 48 && n > 64 && n < 96) return false;
    return wgrad_gather_us(n, cin, cout, chunk_vox) > 14 + (cin < 8 ? 0.55 * ((cout - 1) / 16) : 0);
}

int check_tensor(int n, int ld, int off, int c) {
    if (n < 1 || ld < 1 || off < 0 || c < 1 || off + c > ld)
        return lgdhip::set_error(LGDHIP_ERR_INVALID_ARG, "bad tensor shape (n, ld, off, c)");
    if ((int64_t)n * n * n * ld >= ((int64_t)1 << 40))
        return lgdhip::set_error(LGDHIP_ERR_UNSUPPORTED, "tensor too large");
    return 0;
}

int small_workspace() {
    return lgdhip::set_error(LGDHIP_ERR_WORKSPACE,
                             "forward workspace too small (lgdhip_conv3d_forward_workspace_bytes)");
}

// lgdhip_conv3d_bf16_forward_ws, with the ReLU mask of an activation where the
// launch takes one along (masked_out; lda, offa its row stride and offset)
int conv3d_forward(const void *x, int n, int ldx, int offx, int cin, int ksize, const void *w, const float *bias,
                   int cout, void *y, int ldy, int offy, float *y32, int ld32, int relu, int accumulate,
                   void *workspace, size_t workspace_bytes, const u16 *act, int lda, int offa, bool &masked_out,
                   lgdhip_stream_t stream) {
    masked_out = false;
    LGD_REQUIRE(x && w && (y || y32), "NULL pointer");
    LGD_REQUIRE(ksize == 1 || ksize == 3, "ksize must be 1 or 3");
    LGD_REQUIRE(cout >= 1 && cout <= 16 * kMaxNTiles, "cout must be in [1, 192]");
    LGD_REQUIRE(!y32 || ld32 >= cout, "ld32 must be >= cout");
    int rc = check_tensor(n, ldx, offx, cin);
    if (rc) return rc;
    if (y) {
        rc = check_tensor(n, ldy, offy, cout);
        if (rc) return rc;
    }
    if ((cin & 7) == 0) {
        LGD_REQUIRE((ldx & 7) == 0 && (offx & 7) == 0, "ldx and offx must be multiples of 8 when cin % 8 == 0");
        LGD_REQUIRE(((uintptr_t)x & 15) == 0, "x must be 16-byte aligned");
    }
    LGD_REQUIRE(((uintptr_t)w & 15) == 0, "w must be 16-byte aligned");
    const int Kp = lgdhip_conv3d_kpad(cin, ksize);
    const int nt = (cout + 15) / 16;
    hipStream_t s = lgdhip::as_stream(stream);
    const u16 *X = (const u16 *)x;
    const u16 *Wb = (const u16 *)w;
    u16 *Y = (u16 *)y;
    const int64_t nvox = (int64_t)n * n * n;
    if (ksize == 1 && cout == 1 && (cin & 7) == 0) {  // ldx, offx, alignment checked above
        conv1x1_to1<<<(unsigned)((nvox + 255) / 256), 256, 0, s>>>(X, nvox, ldx, offx, cin, Wb, bias, Y, ldy, offy,
                                                                    y32, ld32, relu, accumulate);
        LGD_LAUNCHED("conv1x1_to1");
        return 0;
    }
    if (ksize == 1 && cin == 1 && cout % 8 == 0 && y && !y32 && !accumulate && (ldy & 7) == 0 && (offy & 7) == 0 &&
        ((uintptr_t)y & 15) == 0 && nvox * (cout / 8) < INT32_MAX) {
        const uint32_t items = (uint32_t)(nvox * (cout / 8));
        masked_out = act && vec8(act, y, cout, lda, offa, ldy, offy);
        conv1x1_from1<<<(unsigned)((items + 255u) / 256u), 256, 0, s>>>(X, items, ldx, offx, Wb, Kp, bias, cout / 8, Y,
                                                                      ldy, offy, relu, masked_out ? act : nullptr, lda,
                                                                      offa);
        LGD_LAUNCHED("conv1x1_from1");
        return 0;
    }
    // z-marching kernel: output channels a multiple of 16, the BF16 output (if
    // any) into an 8-byte aligned range, input of 1 to 8 groups of 8 channels (or
    // a masked row of fewer than 8).  It was the fastest at every such shape
    // measured (figures at the kernel), except that one work-group per CU (7
    // groups on) and two slices lose to the LDS-tile kernel's one pass over 32
    // channels (64^3 64 -> 32: 71 us, there 63).  It keeps the k order of the
    // kernel the layer would go to, so it leaves out the layers that the
    // GEMM-tiled kernel splits more than two ways.
    if (ksize == 3 && cout % 16 == 0 && n >= kLdsMinN && !accumulate &&
        (!y || ((ldy & 3) == 0 && (offy & 3) == 0 && ((uintptr_t)y & 7) == 0))) {
        const bool masked = cin < 8 && (ldx & 7) == 0 && (offx & 7) == 0 && offx + 8 <= ldx &&
                            ((uintptr_t)x & 15) == 0;
        const int groups = (cin & 7) == 0 ? cin / 8 : (masked ? 1 : 0);
        // (with one group the two orders are the same)
        const bool plain = y && !y32 && (ldy & 7) == 0 && (offy & 7) == 0 && ((uintptr_t)y & 15) == 0;
        const bool gemm_order = groups > 1 && (n < kZmGroupOrderN || groups > 6 || !plain) &&
                                gemm_applies(n, cin, ksize, cout);
        int split = 0;
        double gemm_us = 1e300;
        if (gemm_order) {
            const GemmPlan p = gemm_plan(n, cin, cout, workspace != nullptr);
            if (workspace && workspace_bytes < gemm_workspace_bytes(n, p)) return small_workspace();
            split = p.slices;
            gemm_us = 22 + 0.0245 * (double)p.mblocks * p.nblocks;
        }
        const bool fits = groups >= 1 && (groups <= 6 || (groups <= 8 && (split || cout == 16))) && split <= 2;
        const ZmPlan z = fits ? zm_plan(n, groups, cout, masked) : ZmPlan{};
        // 7 groups in tap-major order take 3.15 us a plane step, where 8 take 2.6: the
        // GEMM-tiled kernel keeps the launches that this makes too long (33^3 56 -> 96
        // 62 us, there 46; 96^3 56 -> 64 415, there 365; but 63^3 56 -> 32 60, there 116)
        if (fits && !(groups == 7 && 3.15 * z.steps > gemm_us)) {
            const unsigned wgs = (unsigned)((int64_t)z.bx * z.by * z.bz * z.slices), per = lgdhip::xcd_per(wgs);
            // the mask is compiled for square layers of 16, 32 and 64 channels,
            // those with a ReLU on both sides in a network
            masked_out = act && !y32 && z.nt == 1 && (groups == 2 || groups == 4 || groups == 8) && (lda & 3) == 0 &&
                         (offa & 3) == 0 && ((uintptr_t)act & 7) == 0;
#define LGD_ZM_CASE(G, I, NT, S, M)                                                                         \
    if (groups == G && (I == kInMasked) == masked && z.nt == NT && split == S && M == masked_out)           \
        conv3d_fwd_zm<G, I, NT, S, M><<<lgdhip::xcd_groups(wgs), 256, 0, s>>>(                              \
            X, n, ldx, offx, cin, Wb, Kp, bias, Y, ldy, offy, y32, ld32, relu, act, lda, offa, z.bx, z.by,  \
            z.slices, z.zchunk, wgs, per);
#define LGD_ZM_CASES(G, NT, M)                                                          \
    LGD_ZM_CASE(G, kInVec, NT, 0, M) LGD_ZM_CASE(G, kInVec, NT, 1, M) LGD_ZM_CASE(G, kInVec, NT, 2, M)
            LGD_ZM_CASE(1, kInMasked, 1, 0, false) LGD_ZM_CASE(1, kInMasked, 2, 0, false)
            LGD_ZM_CASE(1, kInMasked, 3, 0, false) LGD_ZM_CASE(1, kInVec, 1, 0, false)
            LGD_ZM_CASE(1, kInVec, 2, 0, false) LGD_ZM_CASE(1, kInVec, 3, 0, false)
            LGD_ZM_CASES(2, 1, false) LGD_ZM_CASES(2, 2, false) LGD_ZM_CASES(3, 1, false) LGD_ZM_CASES(4, 1, false)
            LGD_ZM_CASES(5, 1, false) LGD_ZM_CASES(6, 1, false) LGD_ZM_CASES(7, 1, false) LGD_ZM_CASES(8, 1, false)
            LGD_ZM_CASES(2, 1, true) LGD_ZM_CASES(4, 1, true) LGD_ZM_CASES(8, 1, true)
#undef LGD_ZM_CASES
#undef LGD_ZM_CASE
            LGD_LAUNCHED("conv3d_fwd_zm");
            return 0;
        }
    }
    if (gemm_applies(n, cin, ksize, cout)) {
        const GemmPlan p = gemm_plan(n, cin, cout, workspace != nullptr);
        if (workspace && workspace_bytes < gemm_workspace_bytes(n, p)) return small_workspace();
        const unsigned blocks = (unsigned)((int64_t)p.mblocks * p.nblocks * p.slices);
        if (p.slices > 1) {
            // (gemm_plan splits only launches of fewer than 4 x 256 blocks)
            float *P = (float *)workspace;
            conv3d_fwd_gemm<true><<<blocks, 256, 0, s>>>(X, n, ldx, offx, cin, Wb, Kp, bias, cout, Y, ldy, offy, y32,
                                                         ld32, relu, accumulate, p.mblocks, p.nblocks, p.slices,
                                                         p.stages, P);
            LGD_LAUNCHED("conv3d_fwd_gemm");
            conv3d_gemm_reduce<<<blocks_for(nvox * cout), 256, 0, s>>>(P, nvox, p.nblocks * kGemmBN, p.slices, bias,
                                                                       cout, Y, ldy, offy, y32, ld32, relu,
                                                                       accumulate);
            LGD_LAUNCHED("conv3d_gemm_reduce");
        } else {
            conv3d_fwd_gemm<false><<<blocks, 256, 0, s>>>(X, n, ldx, offx, cin, Wb, Kp, bias, cout, Y, ldy, offy, y32,
                                                          ld32, relu, accumulate, p.mblocks, p.nblocks, 1, p.stages,
                                                          nullptr);
            LGD_LAUNCHED("conv3d_fwd_gemm");
        }
        return 0;
    }
    if (ksize == 3 && nt <= 2 && n >= kLdsMinN) {
        const int bx = (n + kLdsTX - 1) / kLdsTX, by = (n + kLdsTY - 1) / kLdsTY;
        const int bz = (n + 8 / nt - 1) / (8 / nt);
        const unsigned blocks = (unsigned)((int64_t)bx * by * bz);
        // input: 16-byte loads when cin % 8 == 0 (ldx, offx and the alignment
        // were checked above), or for cin < 8 when the 8-channel row
        // [offx, offx + 8) lies inside the voxel's ldx channels and is aligned
        const bool aligned_row = cin < 8 && (ldx & 7) == 0 && (offx & 7) == 0 && offx + 8 <= ldx &&
                                 ((uintptr_t)x & 15) == 0;
        const int in = (cin & 7) == 0 ? kInVec : (aligned_row ? kInMasked : kInElem);
        // output: 16-byte stores of full cout tiles into an aligned slice
        const bool vst = y && !y32 && !accumulate && cout == 16 * nt && (ldy & 7) == 0 && (offy & 7) == 0 &&
                         ((uintptr_t)y & 15) == 0;
#define LGD_LDS_CASE(T, I, V)                                                                                   \
    if (nt == T && in == I && vst == V)                                                                         \
        conv3d_fwd_lds<T, I, V><<<blocks, 256, 0, s>>>(X, n, ldx, offx, cin, Wb, Kp, bias, cout, Y, ldy, offy, y32, \
                                                       ld32, relu, accumulate, bx, by);
        LGD_LDS_CASE(1, kInVec, true) LGD_LDS_CASE(1, kInVec, false) LGD_LDS_CASE(1, kInMasked, true)
        LGD_LDS_CASE(1, kInMasked, false) LGD_LDS_CASE(1, kInElem, true) LGD_LDS_CASE(1, kInElem, false)
        LGD_LDS_CASE(2, kInVec, true) LGD_LDS_CASE(2, kInVec, false) LGD_LDS_CASE(2, kInMasked, true)
        LGD_LDS_CASE(2, kInMasked, false) LGD_LDS_CASE(2, kInElem, true) LGD_LDS_CASE(2, kInElem, false)
#undef LGD_LDS_CASE
        LGD_LAUNCHED("conv3d_fwd_lds");
        return 0;
    }
    const FwdShape sh = fwd_shape(nvox, nt);
#define LGD_CONV_CASE(T, M)                                                                                   \
    if (sh.nt == T && sh.mt == M) {                                                                           \
        const int64_t waves = (nvox + 16 * M - 1) / (16 * M) * sh.groups;                                     \
        conv3d_fwd_mfma<T, M><<<(unsigned)((waves + 3) / 4), 256, 0, s>>>(                                    \
            X, n, ldx, offx, cin, ksize, Wb, Kp, bias, cout, Y, ldy, offy, y32, ld32, relu, accumulate,        \
            sh.groups);                                                                                       \
    }
    LGD_CONV_CASE(1, 4) LGD_CONV_CASE(1, 2) LGD_CONV_CASE(1, 1)
    LGD_CONV_CASE(2, 4) LGD_CONV_CASE(2, 2) LGD_CONV_CASE(2, 1)
    LGD_CONV_CASE(3, 4) LGD_CONV_CASE(3, 2) LGD_CONV_CASE(3, 1)
    LGD_CONV_CASE(4, 4) LGD_CONV_CASE(4, 2) LGD_CONV_CASE(4, 1)
    LGD_CONV_CASE(5, 2) LGD_CONV_CASE(5, 1)
    LGD_CONV_CASE(6, 2) LGD_CONV_CASE(6, 1)
    LGD_CONV_CASE(7, 2) LGD_CONV_CASE(7, 1)
    LGD_CONV_CASE(8, 2) LGD_CONV_CASE(8, 1)
    LGD_CONV_CASE(9, 1)
    LGD_CONV_CASE(10, 1)
    LGD_CONV_CASE(11, 1)
    LGD_CONV_CASE(12, 1)
#undef LGD_CONV_CASE
    LGD_LAUNCHED("conv3d_fwd_mfma");
    return 0;
}

} // namespace

extern "C" {

int lgdhip_conv3d_kpad(int cin, int ksize) { return (((ksize == 1 ? 1 : 27) * cin + 31) / 32) * 32; }

size_t lgdhip_conv3d_forward_workspace_bytes(int n, int cin, int ksize, int cout) {
    if (n < 1 || cin < 1 || cout < 1 || !gemm_applies(n, cin, ksize, cout)) return 0;
    return gemm_workspace_bytes(n, gemm_plan(n, cin, cout, true));
}

int lgdhip_conv3d_bf16_forward(const void *x, int n, int ldx, int offx, int cin, int ksize, const void *w,
                               const float *bias, int cout, void *y, int ldy, int offy, float *y32, int ld32,
                               int relu, int accumulate, lgdhip_stream_t stream) {
    return lgdhip_conv3d_bf16_forward_ws(x, n, ldx, offx, cin, ksize, w, bias, cout, y, ldy, offy, y32, ld32, relu,
                                         accumulate, nullptr, 0, stream);
}

int lgdhip_conv3d_bf16_forward_ws(const void *x, int n, int ldx, int offx, int cin, int ksize, const void *w,
                                  const float *bias, int cout, void *y, int ldy, int offy, float *y32, int ld32,
                                  int relu, int accumulate, void *workspace, size_t workspace_bytes,
                                  lgdhip_stream_t stream) {
    bool masked;
    return conv3d_forward(x, n, ldx, offx, cin, ksize, w, bias, cout, y, ldy, offy, y32, ld32, relu, accumulate,
                          workspace, workspace_bytes, nullptr, 0, 0, masked, stream);
}

int lgdhip_conv3d_bf16_dgrad_relu(const void *x, int n, int ldx, int offx, int cin, int ksize, const void *w, int cout,
                                  void *y, int ldy, int offy, const void *act, int lda, int offa, void *workspace,
                                  size_t workspace_bytes, lgdhip_stream_t stream) {
    LGD_REQUIRE(y && act, "NULL pointer");
    int rc = check_tensor(n, lda, offa, cout);
    if (rc) return rc;
    bool masked;
    rc = conv3d_forward(x, n, ldx, offx, cin, ksize, w, nullptr, cout, y, ldy, offy, nullptr, 0, 0, 0, workspace,
                        workspace_bytes, (const u16 *)act, lda, offa, masked, stream);
    if (rc || masked) return rc;
    return lgdhip_relu_backward_bf16(y, ldy, offy, act, lda, offa, cout, (int64_t)n * n * n, stream);
}

size_t lgdhip_conv3d_wgrad_workspace_bytes(int n, int cin, int ksize, int cout, int chunk_vox) {
    if (n < 1 || cin < 1 || cout < 1 || (ksize != 1 && ksize != 3)) return 0;
    if (chunk_vox <= 0) chunk_vox = wgrad_chunk(n, cin, ksize, cout);
    const int64_t nvox = (int64_t)n * n * n;
    const int64_t chunks = (nvox + chunk_vox - 1) / chunk_vox;
    // [P: chunk partials][bias partials], for whichever kernel the tensors allow
    int64_t partials = chunks;
    if (wgrad_zm_shape(cin, ksize, cout)) partials = std::max<int64_t>(partials, wgrad_zm_plan(n, cin, cout).chunks);
    return (size_t)(partials * cout * lgdhip_conv3d_kpad(cin, ksize) * 4) +
           (size_t)cout * (size_t)((nvox + kBiasChunk - 1) / kBiasChunk) * 4;
}

int lgdhip_conv3d_bf16_wgrad(const void *x, int n, int ldx, int offx, int cin, int ksize, const void *dy, int ldy,
                             int offy, int cout, float *dw, float *db, int accumulate, int chunk_vox,
                             void *workspace, size_t workspace_bytes, lgdhip_stream_t stream) {
    LGD_REQUIRE(x && dy && dw && workspace, "NULL pointer");
    LGD_REQUIRE(ksize == 1 || ksize == 3, "ksize must be 1 or 3");
    LGD_REQUIRE(cout >= 1 && cout <= 16 * kMaxNTiles, "cout must be in [1, 192]");
    int rc = check_tensor(n, ldx, offx, cin);
    if (rc) return rc;
    rc = check_tensor(n, ldy, offy, cout);
    if (rc) return rc;
    if (chunk_vox <= 0) chunk_vox = wgrad_chunk(n, cin, ksize, cout);
    LGD_REQUIRE(chunk_vox % 32 == 0, "chunk_vox must be a multiple of 32");
    if (workspace_bytes < lgdhip_conv3d_wgrad_workspace_bytes(n, cin, ksize, cout, chunk_vox))
        return lgdhip::set_error(LGDHIP_ERR_WORKSPACE, "wgrad workspace too small");
    const int Kp = lgdhip_conv3d_kpad(cin, ksize);
    const int K = (ksize == 1 ? 1 : 27) * cin;
    const int64_t nvox = (int64_t)n * n * n;
    const int chunks = (int)((nvox + chunk_vox - 1) / chunk_vox);
    hipStream_t s = lgdhip::as_stream(stream);
    float *P = (float *)workspace;
    int parts = chunks;
    const bool zm = wgrad_zm_shape(cin, ksize, cout) && ldx % 8 == 0 && offx % 8 == 0 && ldy % 8 == 0 &&
                    offy % 8 == 0 && (cin >= 8 || offx + 8 <= ldx) && (uintptr_t)x % 16 == 0 &&
                    (uintptr_t)dy % 16 == 0 && (int64_t)n * n * std::max(ldx, ldy) < INT32_MAX &&
                    wgrad_columns_pay(n, cin, cout, chunk_vox);
    if (zm) {
        const ZmWgrad w = wgrad_zm_plan(n, cin, cout);
        parts = w.chunks;
        const unsigned groups = (unsigned)w.groups(), per = lgdhip::xcd_per(groups);
#define LGD_ZW_CASE(TI, TO, KS, IN)                                                                            \
    if (w.ti == TI && w.to == TO && w.ks == KS && (cin < 8) == (IN == kInMasked))                              \
        conv3d_wgrad_zm<TI, TO, KS, IN><<<lgdhip::xcd_groups(groups), 64 * TI * TO * KS, 0, s>>>(              \
            (const u16 *)x, n, ldx, offx, cin, (const u16 *)dy, ldy, offy, cout, Kp, w.zchunk, w.bx, w.by,     \
            w.gi, w.go, P, groups, per);
        LGD_ZW_CASE(1, 1, 4, kInVec) LGD_ZW_CASE(1, 2, 4, kInVec) LGD_ZW_CASE(2, 1, 4, kInVec)
        LGD_ZW_CASE(3, 1, 4, kInVec) LGD_ZW_CASE(2, 2, 2, kInVec) LGD_ZW_CASE(3, 2, 1, kInVec)
        LGD_ZW_CASE(2, 4, 1, kInVec) LGD_ZW_CASE(4, 2, 1, kInVec)
        LGD_ZW_CASE(1, 1, 4, kInMasked) LGD_ZW_CASE(1, 2, 4, kInMasked)
#undef LGD_ZW_CASE
        LGD_LAUNCHED("conv3d_wgrad_zm");
    } else if (ksize == 1 && cout == 1 && cin % 8 == 0 && (cin & (cin - 1)) == 0 && ldx % 8 == 0 && offx % 8 == 0 &&
               (uintptr_t)x % 16 == 0 && cin <= 192) {
        conv1x1_to1_wgrad<<<(unsigned)chunks, 256, 0, s>>>((const u16 *)x, nvox, ldx, offx, (const u16 *)dy, ldy, offy,
                                                           cin / 8, Kp, chunk_vox, P);
        LGD_LAUNCHED("conv1x1_to1_wgrad");
    } else {
        const int64_t waves = (int64_t)chunks * (Kp / 16);
        const unsigned wgs = (unsigned)((waves + 3) / 4);
        const unsigned per = lgdhip::xcd_per(wgs), grid = lgdhip::xcd_groups(wgs);
        const int nt = (cout + 15) / 16;
#define LGD_WG_CASE(T)                                                                                       \
    case T:                                                                                                  \
        conv3d_wgrad_mfma<T><<<grid, 256, 0, s>>>((const u16 *)x, n, ldx, offx, cin, ksize, (const u16 *)dy, \
                                                  ldy, offy, cout, Kp, chunk_vox, P, per);                   \
        break;
        switch (nt) {
            LGD_WG_CASE(1)
            LGD_WG_CASE(2)
            LGD_WG_CASE(3)
            LGD_WG_CASE(4)
            LGD_WG_CASE(5)
            LGD_WG_CASE(6)
            LGD_WG_CASE(7)
            LGD_WG_CASE(8)
            LGD_WG_CASE(9)
            LGD_WG_CASE(10)
            LGD_WG_CASE(11)
            LGD_WG_CASE(12)
        }
#undef LGD_WG_CASE
        LGD_LAUNCHED("conv3d_wgrad_mfma");
    }
    const unsigned outs = (unsigned)((cout * Kp + kWgradReduceOutputs - 1) / kWgradReduceOutputs);
    if (outs >= 2 * lgdhip::kCUs || parts <= 16)
        conv3d_wgrad_reduce<4><<<outs, dim3(kWgradReduceOutputs, 4), 0, s>>>(P, parts, cout, Kp, K, dw, accumulate);
    else
        conv3d_wgrad_reduce<16><<<outs, dim3(kWgradReduceOutputs, 16), 0, s>>>(P, parts, cout, Kp, K, dw, accumulate);
    LGD_LAUNCHED("conv3d_wgrad_reduce");
    if (db) {
        const int bchunks = (int)((nvox + kBiasChunk - 1) / kBiasChunk);
        float *Pb = P + (size_t)parts * cout * Kp;
        const u16 *g = (const u16 *)dy;
        const bool rows = cout % 8 == 0 && ldy % 8 == 0 && offy % 8 == 0 && (uintptr_t)dy % 16 == 0;
        if (rows && cout % 16 == 0)
            bias_grad_rows<2><<<dim3(bchunks, cout / 16), 256, 0, s>>>(g, nvox, ldy, offy, Pb, bchunks);
        else if (rows)
            bias_grad_rows<1><<<dim3(bchunks, cout / 8), 256, 0, s>>>(g, nvox, ldy, offy, Pb, bchunks);
        else
            bias_grad_partial<<<bchunks, 256, 0, s>>>(g, nvox, ldy, offy, cout, Pb, bchunks);
        row_sum_final<<<blocks_for(cout), 256, 0, s>>>(Pb, bchunks, cout, db, accumulate);
        LGD_LAUNCHED("bias_grad");
    }
    return 0;
}

int lgdhip_conv3d_dgrad_weights(const void *w, int cin, int cout, int ksize, void *wt, lgdhip_stream_t stream) {
    LGD_REQUIRE(w && wt, "NULL pointer");
    LGD_REQUIRE(ksize == 1 || ksize == 3, "ksize must be 1 or 3");
    const int Kp = lgdhip_conv3d_kpad(cin, ksize);
    const int Kpt = lgdhip_conv3d_kpad(cout, ksize);
    conv3d_dgrad_weights<<<blocks_for((int64_t)cin * Kpt), 256, 0, lgdhip::as_stream(stream)>>>(
        (const u16 *)w, cin, cout, ksize, Kp, (u16 *)wt, Kpt);
    LGD_LAUNCHED("conv3d_dgrad_weights");
    return 0;
}

int lgdhip_relu_backward_bf16(void *g, int ldg, int offg, const void *y, int ldy, int offy, int c, int64_t nvox,
                              lgdhip_stream_t stream) {
    LGD_REQUIRE(g && y && c > 0 && nvox > 0, "bad arguments");
    if (vec8(g, y, c, ldg, offg, ldy, offy) && nvox * (c / 8) < INT32_MAX) {
        const bool dense = ldg == c && ldy == c && offg == 0 && offy == 0;
        const uint32_t items = (uint32_t)(nvox * (c / 8));
        relu_backward_v8<<<blocks_for(items), 256, 0, lgdhip::as_stream(stream)>>>(
            (u16 *)g, ldg, offg, (const u16 *)y, ldy, offy, dense ? 0 : c / 8, items);
        LGD_LAUNCHED("relu_backward_v8");
        return 0;
    }
    relu_backward<<<blocks_for(nvox * c), 256, 0, lgdhip::as_stream(stream)>>>((u16 *)g, ldg, offg, (const u16 *)y,
                                                                               ldy, offy, c, nvox);
    LGD_LAUNCHED("relu_backward");
    return 0;
}

int lgdhip_avgpool2_bf16(const void *x, int n, int ldx, int offx, void *y, int ldy, int offy, int c,
                         lgdhip_stream_t stream) {
    LGD_REQUIRE(x && y && n % 2 == 0, "bad arguments");
    const int64_t m = n / 2;
    if (vec8(x, y, c, ldx, offx, ldy, offy) && n <= kMaxRowGrid) {
        avgpool2_v8<<<row_grid((int)m, c / 8), 256, 0, lgdhip::as_stream(stream)>>>(
            (const u16 *)x, n, ldx, offx, (u16 *)y, ldy, offy, c / 8);
        LGD_LAUNCHED("avgpool2_v8");
        return 0;
    }
    avgpool2<<<blocks_for(m * m * m * c), 256, 0, lgdhip::as_stream(stream)>>>((const u16 *)x, n, ldx, offx, (u16 *)y,
                                                                               ldy, offy, c);
    LGD_LAUNCHED("avgpool2");
    return 0;
}

int lgdhip_avgpool2_backward_bf16(const void *dy, int n, int ldy, int offy, void *dx, int ldx, int offx, int c,
                                  int accumulate, lgdhip_stream_t stream) {
    return lgdhip_avgpool2_backward_relu_bf16(dy, n, ldy, offy, dx, ldx, offx, c, accumulate, nullptr, 0, 0, stream);
}

int lgdhip_avgpool2_backward_relu_bf16(const void *dy, int n, int ldy, int offy, void *dx, int ldx, int offx, int c,
                                       int accumulate, const void *act, int lda, int offa, lgdhip_stream_t stream) {
    LGD_REQUIRE(dy && dx && n % 2 == 0, "bad arguments");
    if (vec8(dy, dx, c, ldy, offy, ldx, offx) && (!act || vec8(act, dx, c, lda, offa, ldx, offx)) && n <= kMaxRowGrid) {
        avgpool2_backward_v8<<<row_grid(n, c / 8), 256, 0, lgdhip::as_stream(stream)>>>(
            (const u16 *)dy, n, ldy, offy, (u16 *)dx, ldx, offx, c / 8, accumulate, (const u16 *)act, lda, offa);
        LGD_LAUNCHED("avgpool2_backward_v8");
        return 0;
    }
    avgpool2_backward<<<blocks_for((int64_t)n * n * n * c), 256, 0, lgdhip::as_stream(stream)>>>(
        (const u16 *)dy, n, ldy, offy, (u16 *)dx, ldx, offx, c, accumulate);
    LGD_LAUNCHED("avgpool2_backward");
    return act ? lgdhip_relu_backward_bf16(dx, ldx, offx, act, lda, offa, c, (int64_t)n * n * n, stream) : 0;
}

int lgdhip_upsample2_bf16(const void *x, int m, int ldx, int offx, void *y, int ldy, int offy, int c,
                          lgdhip_stream_t stream) {
    LGD_REQUIRE(x && y && m >= 1, "bad arguments");
    const int64_t n = 2 * (int64_t)m;
    if (vec8(x, y, c, ldx, offx, ldy, offy) && n <= kMaxRowGrid) {
        upsample2_v8<<<row_grid((int)n, c / 8), 256, 0, lgdhip::as_stream(stream)>>>(
            (const u16 *)x, m, ldx, offx, (u16 *)y, ldy, offy, c / 8);
        LGD_LAUNCHED("upsample2_v8");
        return 0;
    }
    upsample2<<<blocks_for(n * n * n * c), 256, 0, lgdhip::as_stream(stream)>>>((const u16 *)x, m, ldx, offx, (u16 *)y,
                                                                                ldy, offy, c);
    LGD_LAUNCHED("upsample2");
    return 0;
}

int lgdhip_upsample2_concat_bf16(const void *x, int m, int ldx, int offx, int cu, const void *skip, int lds,
                                 int offs, int cs, void *y, int ldy, int offy, lgdhip_stream_t stream) {
    LGD_REQUIRE(x && skip && y && m >= 1 && cu > 0 && cs > 0, "bad arguments");
    const int64_t n = 2 * (int64_t)m;
    if (vec8(x, y, cu, ldx, offx, ldy, offy) && vec8(skip, y, cs, lds, offs, ldy, offy) && n <= kMaxRowGrid) {
        upsample2_concat_v8<<<row_grid((int)n, (cu + cs) / 8), 256, 0, lgdhip::as_stream(stream)>>>(
            (const u16 *)x, m, ldx, offx, cu / 8, (const u16 *)skip, lds, offs, (u16 *)y, ldy, offy, (cu + cs) / 8);
        LGD_LAUNCHED("upsample2_concat_v8");
        return 0;
    }
    upsample2_concat<<<blocks_for(n * n * n * (cu + cs)), 256, 0, lgdhip::as_stream(stream)>>>(
        (const u16 *)x, m, ldx, offx, cu, (const u16 *)skip, lds, offs, cs, (u16 *)y, ldy, offy);
    LGD_LAUNCHED("upsample2_concat");
    return 0;
}

int lgdhip_upsample2_backward_bf16(const void *dy, int m, int ldy, int offy, void *dx, int ldx, int offx, int c,
                                  int accumulate, lgdhip_stream_t stream) {
    return lgdhip_upsample2_backward_relu_bf16(dy, m, ldy, offy, dx, ldx, offx, c, accumulate, nullptr, 0, 0, stream);
}

int lgdhip_upsample2_backward_relu_bf16(const void *dy, int m, int ldy, int offy, void *dx, int ldx, int offx, int c,
                                       int accumulate, const void *act, int lda, int offa, lgdhip_stream_t stream) {
    LGD_REQUIRE(dy && dx && m >= 1, "bad arguments");
    if (vec8(dy, dx, c, ldy, offy, ldx, offx) && (!act || vec8(act, dx, c, lda, offa, ldx, offx)) && 2 * (int64_t)m <= kMaxRowGrid) {
        upsample2_backward_v8<<<row_grid(m, c / 8), 256, 0, lgdhip::as_stream(stream)>>>(
            (const u16 *)dy, m, ldy, offy, (u16 *)dx, ldx, offx, c / 8, accumulate, (const u16 *)act, lda, offa);
        LGD_LAUNCHED("upsample2_backward_v8");
        return 0;
    }
    upsample2_backward<<<blocks_for((int64_t)m * m * m * c), 256, 0, lgdhip::as_stream(stream)>>>(
        (const u16 *)dy, m, ldy, offy, (u16 *)dx, ldx, offx, c, accumulate);
    LGD_LAUNCHED("upsample2_backward");
    return act ? lgdhip_relu_backward_bf16(dx, ldx, offx, act, lda, offa, c, (int64_t)m * m * m, stream) : 0;
}

int lgdhip_pack_bf16(const float *src, int64_t nvox, void *y, int ldy, int offy, lgdhip_stream_t stream) {
    LGD_REQUIRE(src && y && nvox > 0, "bad arguments");
    pack_bf16<<<blocks_for(nvox), 256, 0, lgdhip::as_stream(stream)>>>(src, nvox, (u16 *)y, ldy, offy);
    LGD_LAUNCHED("pack_bf16");
    return 0;
}

int lgdhip_pack_rows_bf16(const float *const *src, int count, int64_t nvox, void *y, int ldy, lgdhip_stream_t stream) {
    LGD_REQUIRE(src && y && nvox > 0 && count >= 1 && count <= 8, "bad arguments");
    LGD_REQUIRE(ldy >= 8 && ldy % 8 == 0 && ((uintptr_t)y & 15) == 0, "rows must be 16-byte aligned, ldy a multiple of 8");
    PackFields f{};
    for (int k = 0; k < count; ++k) {
        LGD_REQUIRE(src[k], "NULL pointer");
        f.f[k] = src[k];
    }
    pack_rows_bf16<<<blocks_for(nvox), 256, 0, lgdhip::as_stream(stream)>>>(f, count, nvox, (u16 *)y, ldy);
    LGD_LAUNCHED("pack_rows_bf16");
    return 0;
}

int64_t lgdhip_mse_partials(int64_t nvox) { return (nvox + 255) / 256; }

int lgdhip_mse_loss(const float *pred, const float *target, int64_t nvox, void *grad, int ldg, float *partial,
                    lgdhip_stream_t stream) {
    LGD_REQUIRE(pred && target && grad && partial && nvox > 0, "bad arguments");
    mse_loss<<<blocks_for(nvox), 256, 0, lgdhip::as_stream(stream)>>>(pred, target, nvox, (u16 *)grad, ldg, partial);
    LGD_LAUNCHED("mse_loss");
    return 0;
}

int lgdhip_adam_step(float *w, float *m, float *v, const float *g, int64_t count, int cols_used, int kp, float lr,
                     float beta1, float beta2, float eps, int t, void *w_bf16, lgdhip_stream_t stream) {
    LGD_REQUIRE(w && m && v && g && count > 0 && t >= 1, "bad arguments");
    const float c1 = 1.0f - powf(beta1, (float)t);
    const float c2 = 1.0f - powf(beta2, (float)t);
    adam_step<<<blocks_for(count), 256, 0, lgdhip::as_stream(stream)>>>(w, m, v, g, count, cols_used, kp, lr, beta1,
                                                                       beta2, eps, c1, c2, (u16 *)w_bf16);
    LGD_LAUNCHED("adam_step");
    return 0;
}

} // extern "C"
