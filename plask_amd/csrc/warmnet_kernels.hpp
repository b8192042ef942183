// Warm-start network kernels: 3x3x3 convolutions on bf16 MFMA (forward, backward
// data, backward weights), pooling / upsampling, the pointwise output head, the
// loss and Adam.  Tensors are channels-last, voxel v = (z * ny + y) * nx + x,
// element [v][c].  All accumulation is fp32.
//
// MFMA v_mfma_f32_16x16x32_bf16 (gfx950), one wave: D(16x16) += A(16x32) B(32x16).
// Lane l supplies row l%16 of A and column l%16 of B, eight k values each (slot
// j of lane group g = l/16 is k = 8g + j on both operands, so any internal k
// order of the instruction gives the same sum), and receives D rows 4g..4g+3 of
// column l%16.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace wn {

typedef __bf16 bf16;
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

struct Vol {
    int nx, ny, nz;
    __host__ __device__ long long n() const { return (long long)nx * ny * nz; }
};

__device__ __forceinline__ float b2f(bf16 v) { return (float)v; }
__device__ __forceinline__ bf16 f2b(float v) { return (bf16)v; }

// Taps: t = (dz + 1) * 9 + (dy + 1) * 3 + (dx + 1); tap 26 - t is the mirrored offset.
//
// Bricks of output voxels: every convolution kernel works on bricks of 16 x 2 YT x 2 ZT
// voxels, whose input (with a halo of one voxel) is staged through LDS once and read from
// there by all 27 taps.
__host__ __device__ inline int ceil_div(int a, int b) { return (a + b - 1) / b; }

// Weights of one layer in the order in which the waves of k_conv3 take them: for input
// channels in chunks of 32 (cin >= 32), tap, group of 16 output channels, lane, the lane's 8
// values (output channel lane % 16, input channels 8 (lane / 16) + 0..7 of the chunk), so
// that a wave reads 1 KiB in a row.  cin = 8: a chunk is 4 taps x 8 channels (lane / 16
// selects the tap; the 28th tap is zero).
__host__ __device__ inline size_t frag_index(int cin, int cout, int tap, int co, int ci) {
    const int nt = cout / 16;
    if (cin == 8) return ((((size_t)(tap >> 2) * nt + (co >> 4)) * 4 + (tap & 3)) * 16 + (co & 15)) * 8 + ci;
    return ((((size_t)(ci >> 5) * 27 + tap) * nt + (co >> 4)) * 4 + ((ci >> 3) & 3)) * 128 + (size_t)(co & 15) * 8 +
           (ci & 7);
}
__host__ __device__ inline size_t frag_size(int cin, int cout) {
    return (size_t)(cin == 8 ? 28 : 27) * cin * cout;
}

// Sizes of the staged input of a brick: half resolution along each axis when the layer's
// nearest upsampling is fused into the load (UP).
template <bool UP, int ZT, int YT> struct Halo {
    static constexpr int X = UP ? 10 : 18;
    static constexpr int Y = UP ? YT + 2 : 2 * YT + 2;
    static constexpr int Z = UP ? ZT + 2 : 2 * ZT + 2;
    static constexpr int N = X * Y * Z;
};

// Copies the input of the brick at (x0, y0, z0) into LDS, channels [c0, c0 + CK) of each
// voxel, zero outside the volume iv; SW: the four 16-byte parts of a voxel's 64 bytes are
// permuted with its x so that 16 lanes reading neighbouring voxels hit different banks.
// STRIDE: bytes per voxel in LDS.
template <bool UP, int ZT, int YT, int CK, int STRIDE, bool SW>
__device__ __forceinline__ void stage_input(const Vol& iv, const bf16* __restrict__ in, int cin, int c0, int x0, int y0,
                                            int z0, unsigned char* lds) {
    using H = Halo<UP, ZT, YT>;
    const int bx = (UP ? x0 >> 1 : x0) - 1, by = (UP ? y0 >> 1 : y0) - 1, bz = (UP ? z0 >> 1 : z0) - 1;
    constexpr int PARTS = CK / 8, TOT = H::N * PARTS;
    constexpr int U = 4;  // loads in flight per thread before their LDS stores
    for (int s0 = threadIdx.x; s0 < TOT; s0 += U * 256) {
        uint4 v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int s = s0 + u * 256;
            const int part = s % PARTS, h = s / PARTS;
            const int hx = h % H::X, hy = (h / H::X) % H::Y, hz = h / (H::X * H::Y);
            const int x = bx + hx, y = by + hy, z = bz + hz;
            v[u] = make_uint4(0u, 0u, 0u, 0u);
            if (s < TOT && (unsigned)x < (unsigned)iv.nx && (unsigned)y < (unsigned)iv.ny && (unsigned)z < (unsigned)iv.nz)
                v[u] = *reinterpret_cast<const uint4*>(in + (((size_t)z * iv.ny + y) * iv.nx + x) * cin + c0 + part * 8);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int s = s0 + u * 256;
            const int part = s % PARTS, h = s / PARTS;
            const int hx = h % H::X;
            const int pp = SW ? part ^ ((hx >> 2) & 3) : part;
            if (s < TOT) *reinterpret_cast<uint4*>(lds + h * STRIDE + pp * 16) = v[u];
        }
    }
}

// Output-stationary 3x3x3 convolution.  A block of 4 waves takes a brick of 16 x 2 YT x 2 ZT
// voxels and 16 CONV_NT output channels; a wave takes ZT x YT of the brick's x rows (16 voxels
// each) and keeps their accumulators in registers.  Input channels go in chunks of 32
// through LDS; per chunk and x offset the wave holds all the input rows its outputs touch
// ((ZT + 2) x (YT + 2), or half of that with the upsampling, where several taps of one
// output row fall on the same input row) in registers and uses each for up to 9 taps.
// w: fragment order (frag_index).  Epilogue: + bias[co] (nullable) + skip[v][co] (nullable),
// ReLU if RELU, bf16 store, 4 channels (8 bytes) per lane and row.
// What bounds it: the matrix cores and the instructions around them.  The earlier kernel
// (one wave per 16 voxels, both operands from global memory for every tap) was held by L1:
// each input value was fetched 27 times and all weights once per 16 voxels.  At 64 x 64 x
// 128 voxels, before and after: 64 -> 32 channels upsampled 523 -> 65 us (0.89 PFLOP/s),
// 128 -> 64 upsampled 228 -> 42 us, 8 -> 32 30 -> 22 us, 32 -> 64 backward data 247 -> 82 us.
// 32 output channels per block: with 64 the last of these took 88 us, a training step of 128 x 128
// x 256 voxels 4.45 instead of 4.30 ms, and no size gained (twice the accumulators: one wave per
// SIMD instead of two).
constexpr int CONV_NT = 2;
template <int CIN, int ZT, int YT, bool UP, bool RELU>
__global__ __launch_bounds__(256) void k_conv3(Vol o, const bf16* __restrict__ in, const bf16* __restrict__ w,
                                               const float* __restrict__ bias, const bf16* __restrict__ skip,
                                               bf16* __restrict__ out, int cout) {
    using H = Halo<UP, ZT, YT>;
    constexpr int NT = CONV_NT;
    constexpr int CK = CIN < 32 ? CIN : 32;
    __shared__ __align__(16) unsigned char tile[H::N * CK * 2];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r = lane & 15, g = lane >> 4;
    const int bxn = ceil_div(o.nx, 16), byn = ceil_div(o.ny, 2 * YT);
    const int b = blockIdx.x;
    const int x0 = (b % bxn) * 16, y0 = (b / bxn) % byn * 2 * YT, z0 = b / (bxn * byn) * 2 * ZT;
    const int nt0 = blockIdx.y * NT, ntall = cout / 16;
    const int wz = (wave >> 1) * ZT, wy = (wave & 1) * YT;  // the wave's rows within the brick
    const Vol iv = UP ? Vol{o.nx >> 1, o.ny >> 1, o.nz >> 1} : o;
    f32x4 acc[ZT * YT][NT];
#pragma unroll
    for (int m = 0; m < ZT * YT; ++m)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    // each lane's byte offset within the weights of one (chunk, tap)
    const bf16* wl = w + ((size_t)nt0 * 64 + lane) * 8;
    if constexpr (CIN == 8) {
        stage_input<UP, ZT, YT, 8, 16, false>(iv, in, CIN, 0, x0, y0, z0, tile);
        __syncthreads();
        const unsigned char* base = tile + ((wz * H::Y + wy) * H::X + r) * 16;
#pragma unroll
        for (int kc = 0; kc < 7; ++kc) {
            const int tap = min(4 * kc + g, 26);  // the 28th tap has zero weights
            const int off = ((tap / 9) * H::Y + (tap / 3) % 3) * H::X + tap % 3;
            bf16x8 bw[NT];
#pragma unroll
            for (int t = 0; t < NT; ++t)
                bw[t] = *reinterpret_cast<const bf16x8*>(wl + ((size_t)kc * ntall + t) * 512);
#pragma unroll
            for (int m = 0; m < ZT * YT; ++m) {
                const bf16x8 a = *reinterpret_cast<const bf16x8*>(base + (off + ((m / YT) * H::Y + m % YT) * H::X) * 16);
#pragma unroll
                for (int t = 0; t < NT; ++t)
                    acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bw[t], a, acc[m][t], 0, 0, 0);
            }
        }
    } else {
        constexpr int ZR = UP ? ZT / 2 + 2 : ZT + 2, YR = UP ? YT / 2 + 2 : YT + 2;  // input rows of a wave
        int loff[3];
#pragma unroll
        for (int dx = 0; dx < 3; ++dx) {
            const int hx = UP ? ((r + dx - 1) >> 1) + 1 : r + dx;
            loff[dx] = hx * 64 + ((g ^ ((hx >> 2) & 3)) << 4);
        }
        const unsigned char* base = tile + ((UP ? wz / 2 : wz) * H::Y + (UP ? wy / 2 : wy)) * (H::X * 64);
        for (int c = 0; c < CIN / 32; ++c) {
            if (c) __syncthreads();
            stage_input<UP, ZT, YT, 32, 64, true>(iv, in, CIN, 32 * c, x0, y0, z0, tile);
            __syncthreads();
            const bf16* wc = wl + (size_t)c * 27 * ntall * 512;
#pragma unroll
            for (int dx = 0; dx < 3; ++dx) {
                bf16x8 row[ZR][YR];
#pragma unroll
                for (int a = 0; a < ZR; ++a)
#pragma unroll
                    for (int q = 0; q < YR; ++q)
                        row[a][q] = *reinterpret_cast<const bf16x8*>(base + (a * H::Y + q) * (H::X * 64) + loff[dx]);
#pragma unroll
                for (int dz = 0; dz < 3; ++dz)
#pragma unroll
                    for (int dy = 0; dy < 3; ++dy) {
                        const int tap = dz * 9 + dy * 3 + dx;
                        bf16x8 bw[NT];
#pragma unroll
                        for (int t = 0; t < NT; ++t)
                            bw[t] = *reinterpret_cast<const bf16x8*>(wc + ((size_t)tap * ntall + t) * 512);
#pragma unroll
                        for (int m = 0; m < ZT * YT; ++m) {
                            // input row of output row m: floor((offset - 1 + tap) / 2) + 1 at half resolution
                            const int za = UP ? (m / YT + dz + 1) >> 1 : m / YT + dz;
                            const int ya = UP ? (m % YT + dy + 1) >> 1 : m % YT + dy;
#pragma unroll
                            for (int t = 0; t < NT; ++t)
                                acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bw[t], row[za][ya], acc[m][t], 0, 0, 0);
                        }
                    }
            }
        }
    }
    // D rows 4g + i: output channels, column r: voxel x0 + r
    const int x = x0 + r;
    f32x4 bb[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) bb[t][i] = bias ? bias[16 * (nt0 + t) + 4 * g + i] : 0.f;
#pragma unroll
    for (int m = 0; m < ZT * YT; ++m) {
        const int y = y0 + wy + m % YT, z = z0 + wz + m / YT;
        if (x >= o.nx || y >= o.ny || z >= o.nz) continue;
        const size_t v = ((size_t)z * o.ny + y) * o.nx + x;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const size_t at = v * cout + 16 * (nt0 + t) + 4 * g;
            bf16x4 sk, res;
            if (skip) sk = *reinterpret_cast<const bf16x4*>(skip + at);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float s = acc[m][t][i] + bb[t][i];
                if (skip) s += b2f(sk[i]);
                if (RELU) s = fmaxf(s, 0.f);
                res[i] = f2b(s);
            }
            *reinterpret_cast<bf16x4*>(out + at) = res;
        }
    }
}

// 4 (voxel) x 16 (channel) block of bf16 in LDS, transposed on the way into registers: the 16
// lanes of a group address 4 channels (8 bytes) each, lane t those of voxel t / 4 and channels
// 4 (t % 4) + 0..3; lane t receives channel t of the 4 voxels.
__device__ __forceinline__ bf16x4 lds_read_tr(const unsigned char* p) {
    typedef __attribute__((address_space(3))) bf16x4* lptr;
    return __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lptr)(p));
}
__device__ __forceinline__ bf16x8 join8(bf16x4 a, bf16x4 b) { return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7); }

// Geometry of the weight-gradient kernel: CB input channels per block (16 per wave; fewer
// than 64 leaves waves that split the voxels: KS of them), bricks of 16 x 2 YT x 4 voxels.
template <int CIN, bool UP> struct WGrad {
    static constexpr int CB = CIN < 64 ? CIN : 64;
    static constexpr int CT = CB < 16 ? 1 : CB / 16;  // channel tiles of a block
    static constexpr int KS = 4 / CT;                 // waves that share a channel tile
    static constexpr int YT = (CB == 64 && !UP) ? 2 : 4;
    static constexpr int SX = CB * 2 + (CB == 64 ? 16 : 0);  // LDS bytes per input voxel
    static constexpr int SG = 64 + 16;                       // and per voxel of 32 gradient channels
    static constexpr int NF = CIN == 8 ? 18 : 27;            // input fragments per 32 voxels
};

// Weight gradient gw[tap][co][ci] = sum_v gy[v][co] x[v + off(tap)][ci] and bias gradient
// gb[co] = sum_v gy[v][co] of one layer: a matrix product over the voxels (32 per MFMA).  A
// block takes 32 output and CB input channels (blockIdx.y) and every gridDim.x-th brick; the
// brick's gradient and input (with halo) are staged channels-last in LDS, and both operands
// are read through the transposing LDS load, which gives a lane 8 voxels of one channel, so
// the 27 taps are address offsets into the same tile.  Accumulators (2 x 27 tiles per wave)
// stay in registers over all its bricks; the block's sums go to its slot of `part`
// ([slot][27 cout cin + cout]) and k_wgrad_reduce adds the slots in a fixed order.
// CIN = 8: 16 columns are two x-neighbouring taps.  UP: x at half resolution.
// What bounds it: LDS reads and matrix cores, about evenly (54 transposed reads for 54
// MFMAs).  The earlier kernel gathered every operand value with a 2-byte load and added
// each wave's tile to memory by atomics; the 64 -> 32 channel layer at 64 x 64 x 128 voxels
// took 4.2 ms, now 82 us and 16 us for the sum of its slots.
template <int CIN, bool UP>
__global__ __launch_bounds__(256, 1) void k_conv3_wgrad(Vol o, const bf16* __restrict__ gy, const bf16* __restrict__ x,
                                                        float* __restrict__ part, int cout) {
    using G = WGrad<CIN, UP>;
    constexpr int YT = G::YT, ZT = 2;
    using H = Halo<UP, ZT, YT>;
    constexpr int BV = 16 * 2 * YT * 2 * ZT;  // voxels of a brick
    __shared__ __align__(16) unsigned char xt[H::N * G::SX + 32];
    __shared__ __align__(16) unsigned char gt[BV * G::SG];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int t16 = lane & 15, g = lane >> 4;
    const int ct = wave % G::CT, ks = wave / G::CT;
    const int cog = blockIdx.y % (cout / 32), cig = blockIdx.y / (cout / 32);
    const Vol iv = UP ? Vol{o.nx >> 1, o.ny >> 1, o.nz >> 1} : o;
    const int bxn = ceil_div(o.nx, 16), byn = ceil_div(o.ny, 2 * YT), bzn = ceil_div(o.nz, 2 * ZT);
    f32x4 acc[G::NF][2], accb[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        accb[c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int f = 0; f < G::NF; ++f) acc[f][c] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    bf16x8 ones;
#pragma unroll
    for (int j = 0; j < 8; ++j) ones[j] = f2b(1.f);
    // The 32 voxels of a step: rows y and y + 1 of the brick; lane group g holds x = 8 (g & 1) +
    // 0..7 of row y + (g >> 1), in two reads of 4 voxels.  Byte offsets of this lane's reads:
    const int py = g >> 1, px = 8 * (g & 1) + (t16 >> 2);
    int goff[2], xoff[2][3][3];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        goff[h] = (16 * py + px + 4 * h) * G::SG + 8 * (t16 & 3);
#pragma unroll
        for (int dy = 0; dy < 3; ++dy)
#pragma unroll
            for (int dx = 0; dx < 3; ++dx) {
                const int hx = UP ? ((px + 4 * h + dx - 1) >> 1) + 1 : px + 4 * h + dx;
                const int hy = UP ? ((py + dy - 1) >> 1) + 1 : py + dy;
                xoff[h][dy][dx] = (hy * H::X + hx) * G::SX + ct * 32 + 8 * (t16 & 3);
            }
    }
    const int nb = bxn * byn * bzn;
    for (int b = blockIdx.x; b < nb; b += gridDim.x) {
        const int x0 = (b % bxn) * 16, y0 = (b / bxn) % byn * 2 * YT, z0 = b / (bxn * byn) * 2 * ZT;
        __syncthreads();
        stage_input<UP, ZT, YT, G::CB, G::SX, false>(iv, x, CIN, cig * G::CB, x0, y0, z0, xt);
        for (int s = threadIdx.x; s < BV * 4; s += 256) {  // 32 gradient channels per voxel
            const int q = s & 3, v = s >> 2;
            const int vx = x0 + (v & 15), vy = y0 + (v >> 4) % (2 * YT), vz = z0 + (v >> 4) / (2 * YT);
            uint4 u = make_uint4(0u, 0u, 0u, 0u);
            if (vx < o.nx && vy < o.ny && vz < o.nz)
                u = *reinterpret_cast<const uint4*>(gy + (((size_t)vz * o.ny + vy) * o.nx + vx) * cout + cog * 32 + 8 * q);
            *reinterpret_cast<uint4*>(gt + v * G::SG + q * 16) = u;
        }
        __syncthreads();
#pragma unroll 1
        for (int st = ks; st < YT * 2 * ZT; st += G::KS) {
            const int yy = 2 * (st % YT), zz = st / YT;  // yy even
            const unsigned char* gp = gt + (zz * 2 * YT + yy) * 16 * G::SG;
            bf16x8 a[2];
#pragma unroll
            for (int c = 0; c < 2; ++c) a[c] = join8(lds_read_tr(gp + goff[0] + 32 * c), lds_read_tr(gp + goff[1] + 32 * c));
#pragma unroll
            for (int c = 0; c < 2; ++c) accb[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[c], ones, accb[c], 0, 0, 0);
#pragma unroll
            for (int dz = 0; dz < 3; ++dz) {
                const int hz = UP ? ((zz + dz - 1) >> 1) + 1 : zz + dz;
                const unsigned char* xp = xt + ((UP ? yy >> 1 : yy) + hz * H::Y) * (H::X * G::SX);
#pragma unroll
                for (int dy = 0; dy < 3; ++dy)
#pragma unroll
                    for (int dx = 0; dx < (CIN == 8 ? 2 : 3); ++dx) {
                        // CIN = 8: columns 8-15 are the next voxel, i.e. the tap at dx + 1
                        const int dd = CIN == 8 ? 2 * dx : dx, f = (dz * 3 + dy) * (CIN == 8 ? 2 : 3) + dx;
                        const bf16x8 bx = join8(lds_read_tr(xp + xoff[0][dy][dd]), lds_read_tr(xp + xoff[1][dy][dd]));
#pragma unroll
                        for (int c = 0; c < 2; ++c)
                            acc[f][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[c], bx, acc[f][c], 0, 0, 0);
                    }
            }
        }
    }
    // D rows 4g + i: output channel, column t16: input channel (CIN = 8: tap dx + t16 / 8)
    float* p = part + (size_t)(blockIdx.x * G::KS + ks) * ((size_t)27 * cout * CIN + cout);
#pragma unroll
    for (int f = 0; f < G::NF; ++f)
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int co = cog * 32 + c * 16 + 4 * g + i;
                if (CIN == 8) {
                    const int dx = 2 * (f & 1) + (t16 >> 3), tap = (f >> 1) * 3 + dx;
                    if (dx < 3) p[((size_t)tap * cout + co) * CIN + (t16 & 7)] = acc[f][c][i];
                } else {
                    p[((size_t)f * cout + co) * CIN + cig * G::CB + ct * 16 + t16] = acc[f][c][i];
                }
            }
    if (cig == 0 && ct == 0 && t16 == 0)
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int i = 0; i < 4; ++i) p[(size_t)27 * cout * CIN + cog * 32 + c * 16 + 4 * g + i] = accb[c][i];
}

// g[e] += the sum over the slots of part ([slot][n]); n weights and biases of a layer lie in
// a row in the parameter vector.  Sixteen threads share an element's slots (up to 1024 slots
// for the few weights of the first layer).
__global__ __launch_bounds__(256) void k_wgrad_reduce(int slots, int n, const float* __restrict__ part,
                                                      float* __restrict__ g) {
    __shared__ float red[16][17];
    const int c = threadIdx.x & 15, q = threadIdx.x >> 4;
    const int e = blockIdx.x * 16 + c;
    float s = 0.f;
    if (e < n)
        for (int k = q; k < slots; k += 16) s += part[(size_t)k * n + e];
    red[q][c] = s;
    __syncthreads();
    if (q == 0 && e < n) {
        float t = 0.f;
#pragma unroll
        for (int k = 0; k < 16; ++k) t += red[k][c];
        g[e] += t;
    }
}

// The kernels between the convolutions take 8 channels (16 bytes) per thread; c: channels,
// a multiple of 8.  They are held by HBM (or latency on the coarser levels).
__device__ __forceinline__ void split8(long long i, int c, const Vol& o, int& c0, int& x, int& y, int& z) {
    const unsigned u = (unsigned)i, per = (unsigned)c / 8, v = u / per, row = v / (unsigned)o.nx;
    c0 = (int)(u - v * per) * 8;
    x = (int)(v - row * (unsigned)o.nx);
    z = (int)(row / (unsigned)o.ny);
    y = (int)(row - (unsigned)z * (unsigned)o.ny);
}

// sums of the 8 children of a half-resolution voxel
__device__ __forceinline__ void children8(const Vol& half, const bf16* __restrict__ full, int c, int c0, int x, int y,
                                          int z, float (&s)[8]) {
    const int fx = 2 * half.nx, fy = 2 * half.ny;
    bf16x8 v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k)
        v[k] = *reinterpret_cast<const bf16x8*>(
            full + (((size_t)(2 * z + (k >> 2)) * fy + (2 * y + ((k >> 1) & 1))) * fx + 2 * x + (k & 1)) * c + c0);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        s[j] = 0.f;
#pragma unroll
        for (int k = 0; k < 8; ++k) s[j] += b2f(v[k][j]);
    }
}

// Backward data through an upsampled input: gx at half resolution is the sum of
// the gradients of its 8 children, zero where the ReLU output relu_of is.  gfull: [V][c] at
// full resolution.
__global__ void k_up_bwd(Vol half, const bf16* __restrict__ gfull, bf16* __restrict__ ghalf, int c,
                         const bf16* __restrict__ relu_of) {
    const long long n = half.n() * (c / 8);
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        int c0, x, y, z;
        split8(i, c, half, c0, x, y, z);
        float s[8];
        const bf16x8 e = *reinterpret_cast<const bf16x8*>(relu_of + i * 8);
        children8(half, gfull, c, c0, x, y, z, s);
        bf16x8 r;
#pragma unroll
        for (int j = 0; j < 8; ++j) r[j] = f2b(b2f(e[j]) > 0.f ? s[j] : 0.f);
        *reinterpret_cast<bf16x8*>(ghalf + i * 8) = r;
    }
}

// 2x2x2 average pooling: out (half resolution) = mean of the 8 children.
__global__ void k_pool(Vol half, const bf16* __restrict__ in, bf16* __restrict__ out, int c) {
    const long long n = half.n() * (c / 8);
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        int c0, x, y, z;
        split8(i, c, half, c0, x, y, z);
        float s[8];
        children8(half, in, c, c0, x, y, z, s);
        bf16x8 r;
#pragma unroll
        for (int j = 0; j < 8; ++j) r[j] = f2b(0.125f * s[j]);
        *reinterpret_cast<bf16x8*>(out + i * 8) = r;
    }
}

// Gradient into a ReLU output e that feeds both a skip connection (gradient
// gskip, full resolution) and a 2x2x2 pool (gradient gpool at half resolution):
// gpre = (gskip + gpool[parent] / 8) * (e > 0); gpre may be gskip.
__global__ void k_skip_pool_bwd(Vol full, const bf16* gskip, const bf16* __restrict__ gpool,
                                const bf16* __restrict__ e, bf16* gpre, int c) {
    const long long n = full.n() * (c / 8);
    const int hx = full.nx >> 1, hy = full.ny >> 1;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        int c0, x, y, z;
        split8(i, c, full, c0, x, y, z);
        const bf16x8 gs = *reinterpret_cast<const bf16x8*>(gskip + i * 8);
        const bf16x8 ev = *reinterpret_cast<const bf16x8*>(e + i * 8);
        const bf16x8 gp = *reinterpret_cast<const bf16x8*>(gpool + (((size_t)(z >> 1) * hy + (y >> 1)) * hx + (x >> 1)) * c + c0);
        bf16x8 r;
#pragma unroll
        for (int j = 0; j < 8; ++j) r[j] = f2b(b2f(ev[j]) > 0.f ? b2f(gs[j]) + 0.125f * b2f(gp[j]) : 0.f);
        *reinterpret_cast<bf16x8*>(gpre + i * 8) = r;
    }
}

// Output head y[v] = sum_c d[v][c] h[c] + hb (32 channels), fp32 out.
__global__ void k_head(long long nv, const bf16* __restrict__ d, const float* __restrict__ h, const float* __restrict__ hb,
                       float* __restrict__ y) {
    for (long long v = (long long)blockIdx.x * blockDim.x + threadIdx.x; v < nv; v += (long long)gridDim.x * blockDim.x) {
        const bf16x8* p = reinterpret_cast<const bf16x8*>(d + v * 32);
        float s = hb[0];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const bf16x8 u = p[q];
#pragma unroll
            for (int j = 0; j < 8; ++j) s += b2f(u[j]) * h[8 * q + j];
        }
        y[v] = s;
    }
}

// Loss, with e = y - t and m = mask (1 when null):
//   L = [sum_v m_v e_v^2 + lambda sum_{x,y edges} (e_a - e_b)^2] / sum_v m_v
//       + sum_{z edges} w_v (e_v - e_{v+z})^2
// where the z-edge weight w_v is per node (edge v -- v + nx ny; null: lambda / sum m).
// gy = dL/dy.  Neighbour differences weight the errors that enlarge the residual of a
// start vector; weights proportional to the vertical conductances make the z term the
// energy of the error in the dominant couplings.
__global__ void k_loss(Vol o, const float* __restrict__ y, const float* __restrict__ t, const float* __restrict__ mask,
                       const float* __restrict__ wz, float inv_norm, float lambda, float* __restrict__ gy,
                       double* __restrict__ loss) {
    __shared__ float red[8];
    const long long nv = o.n();
    float ll = 0.f;
    for (long long v = (long long)blockIdx.x * blockDim.x + threadIdx.x; v < nv; v += (long long)gridDim.x * blockDim.x) {
        const int x = (int)(v % o.nx), yy = (int)((v / o.nx) % o.ny), z = (int)(v / ((long long)o.nx * o.ny));
        const float m = mask ? mask[v] : 1.f;
        const float e = y[v] - t[v];
        float g = 2.f * m * e * inv_norm;
        float l = m * e * e * inv_norm;
        const long long sx = 1, sy = o.nx, sz = (long long)o.nx * o.ny;
        const float lx = lambda * inv_norm;
        if (lambda != 0.f) {
            if (x > 0) g += 2.f * lx * (e - (y[v - sx] - t[v - sx]));
            if (x < o.nx - 1) {
                const float d = e - (y[v + sx] - t[v + sx]);
                g += 2.f * lx * d;
                l += lx * d * d;
            }
            if (yy > 0) g += 2.f * lx * (e - (y[v - sy] - t[v - sy]));
            if (yy < o.ny - 1) {
                const float d = e - (y[v + sy] - t[v + sy]);
                g += 2.f * lx * d;
                l += lx * d * d;
            }
        }
        if (z > 0) {
            const float w = wz ? wz[v - sz] : lx;
            g += 2.f * w * (e - (y[v - sz] - t[v - sz]));
        }
        if (z < o.nz - 1) {
            const float w = wz ? wz[v] : lx;
            const float d = e - (y[v + sz] - t[v + sz]);
            g += 2.f * w * d;
            l += w * d * d;
        }
        gy[v] = g;
        ll += l;
    }
    for (int off = 32; off > 0; off >>= 1) ll += __shfl_xor(ll, off, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ll;
    __syncthreads();
    if (threadIdx.x == 0) {
        float s2 = 0.f;
        for (int k = 0; k < (int)(blockDim.x >> 6); ++k) s2 += red[k];
        atomicAdd(loss, (double)s2);
    }
}

// Head backward: gpre[v][c] = gy_v h_c (d[v][c] > 0); gh[c] += sum_v gy_v d[v][c];
// ghb += sum_v gy_v.  Four lanes per voxel, 8 of the 32 channels each.  Few blocks: each ends
// with 33 atomics on the same 33 addresses (1024 blocks 47 us, 256 blocks and this layout 20).
__global__ __launch_bounds__(256) void k_head_bwd(long long nv, const float* __restrict__ gy, const bf16* __restrict__ d,
                                                  const float* __restrict__ h, bf16* __restrict__ gpre,
                                                  float* __restrict__ gh, float* __restrict__ ghb) {
    __shared__ float red[33][4];
    const int part = threadIdx.x & 3;
    float lh[8], hc[8], lb = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        lh[j] = 0.f;
        hc[j] = h[8 * part + j];
    }
    const long long n4 = nv * 4;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += (long long)gridDim.x * blockDim.x) {
        const float g = gy[i >> 2];
        lb += g;
        const bf16x8 u = *reinterpret_cast<const bf16x8*>(d + i * 8);
        bf16x8 o;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float dv = b2f(u[j]);
            lh[j] += g * dv;
            o[j] = f2b(dv > 0.f ? g * hc[j] : 0.f);
        }
        *reinterpret_cast<bf16x8*>(gpre + i * 8) = o;
    }
    // sums over the 16 voxels of a wave (lanes of equal part), then over the waves
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    auto vsum = [](float v) {
        for (int o = 32; o >= 4; o >>= 1) v += __shfl_xor(v, o, 64);
        return v;
    };
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float s = vsum(lh[j]);
        if (lane < 4) red[8 * lane + j][wid] = s;
    }
    lb = vsum(lb);
    if (lane == 0) red[32][wid] = lb;
    __syncthreads();
    if (threadIdx.x < 33) {
        const float s = (red[threadIdx.x][0] + red[threadIdx.x][1]) + (red[threadIdx.x][2] + red[threadIdx.x][3]);
        if (threadIdx.x < 32) atomicAdd(&gh[threadIdx.x], s);
        else atomicAdd(ghb, s);
    }
}

// Adam (Kingma & Ba 2015) on the fp32 master parameters; bias corrections c1 =
// 1 / (1 - b1^t), c2 = 1 / (1 - b2^t) from the host.
__global__ void k_adam(long long n, float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m,
                       float* __restrict__ v, float lr, float b1, float b2, float eps, float c1, float c2, float gscale) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        const float gi = g[i] * gscale;
        const float mi = b1 * m[i] + (1.f - b1) * gi;
        const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
        m[i] = mi;
        v[i] = vi;
        p[i] -= lr * (mi * c1) / (sqrtf(vi * c2) + eps);
    }
}

// bf16 kernel copies of one conv layer's master weights w[27][cout][cin], in fragment order
// (frag_index): wf = w (forward), wt = the backward-data layer, cout -> cin channels with
// the tap mirrored.
__global__ void k_prep_weights(const float* __restrict__ w, int cout, int cin, bf16* __restrict__ wf,
                               bf16* __restrict__ wt) {
    const long long n = 27LL * cout * cin;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        const int ci = (int)(i % cin);
        const int co = (int)((i / cin) % cout);
        const int t = (int)(i / ((long long)cin * cout));
        const bf16 b = f2b(w[i]);
        wf[frag_index(cin, cout, t, co, ci)] = b;
        if (wt) wt[frag_index(cout, cin, 26 - t, ci, co)] = b;
        if (cin == 8 && t == 26) wf[frag_index(cin, cout, 27, co, ci)] = f2b(0.f);
    }
}

__global__ void k_f32_to_bf16(long long n, const float* __restrict__ a, bf16* __restrict__ b) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        b[i] = f2b(a[i]);
}

__global__ void k_zero_f32(long long n, float* __restrict__ a) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        a[i] = 0.f;
}

__global__ void k_zero_f64(long long n, double* __restrict__ a) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        a[i] = 0.;
}

}  // namespace wn
