// Kernels of the pressure warm-start U-Net (unet.{h,cpp}).
//
// Tensors are channels-last (voxel-major, channel innermost) at the
// resolution of their level, without ghost cells.  Activations and weights
// are BF16 (raw bit patterns, round-to-nearest-even), gradients FP32 (rounded
// to BF16 as matrix operands), and every product accumulates in FP32.  The
// 3x3x3 convolutions with 16 or more channels on both sides, forward and
// backward, are implicit GEMMs on v_mfma_f32_16x16x32_bf16 with register
// tiles per wavefront (k_conv_fwd, k_conv_up_dgrad, k_conv_wgrad); the weight
// gradients of the two end layers, whose inputs are FP32 on one side, run on
// v_mfma_f32_16x16x4_f32.  Operand layouts:
//   16x16x32 BF16, A (rows m) and B (columns n): lane l holds row or column
//     l%16 and eight k values; both operands give a lane's slot the same k,
//     so their order does not change the sum
//   16x16x4 FP32, A and B: lane l holds row or column l%16, k = l/16
//   D (16x16 FP32): lane l holds D[4*(l/16) .. +3][l%16]
//
// Sums over voxels (weight and bias gradients, the loss) go to one partial
// row per workgroup, and one launch adds the rows in a fixed order
// (k_sum_rows): the gradients are the same bits in every run.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <algorithm>
#include <stdexcept>
#include <type_traits>

#include "unet_kernels.h"

namespace artss {
namespace nn {

namespace {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ inline float bf2f(uint16_t b) { return __uint_as_float(static_cast<unsigned>(b) << 16); }
__device__ inline uint16_t f2bf(float f) {
    unsigned u = __float_as_uint(f);
    u += 0x7FFFu + ((u >> 16) & 1u);  // round to nearest even (finite inputs)
    return static_cast<uint16_t>(u >> 16);
}
// whether a BF16 bit pattern is > 0
__device__ inline bool positive(unsigned b) { return __uint_as_float(b << 16) > 0.f; }
__device__ inline unsigned pack2(float lo, float hi) {
    return static_cast<unsigned>(f2bf(lo)) | (static_cast<unsigned>(f2bf(hi)) << 16);
}

__device__ inline long long vox(const Dims &D, int x, int y, int z) {
    return (static_cast<long long>(z) * D.Y + y) * D.X + x;
}

__device__ inline void tap_offset(int t, int &dx, int &dy, int &dz) {
    dz = t / 9 - 1;
    dy = (t / 3) % 3 - 1;
    dx = t % 3 - 1;
}

// The four channels a lane holds of an output voxel, at element o of the
// output: bias, activation and skip as one 8-byte write (pre: also before
// the activation), or with GRAD the FP32 sums, zero where the BF16 activation
// `skip` (optional) is not positive
template <bool GRAD>
__device__ __forceinline__ void store_tile(const f32x4 &acc, const float *bias, long long o, uint16_t *__restrict__ out,
                                           uint16_t *__restrict__ pre, const uint16_t *__restrict__ skip, int relu,
                                           float *__restrict__ gin) {
    if (GRAD) {
        float4 g{acc[0], acc[1], acc[2], acc[3]};
        if (skip) {
            const uint2 m = *reinterpret_cast<const uint2 *>(skip + o);
            g.x = positive(m.x & 0xFFFFu) ? g.x : 0.f;
            g.y = positive(m.x >> 16) ? g.y : 0.f;
            g.z = positive(m.y & 0xFFFFu) ? g.z : 0.f;
            g.w = positive(m.y >> 16) ? g.w : 0.f;
        }
        *reinterpret_cast<float4 *>(gin + o) = g;
        return;
    }
    float c4[4], r[4];
#pragma unroll
    for (int e = 0; e < 4; e++) c4[e] = acc[e] + bias[e];
    if (pre) *reinterpret_cast<uint2 *>(pre + o) = uint2{pack2(c4[0], c4[1]), pack2(c4[2], c4[3])};
#pragma unroll
    for (int e = 0; e < 4; e++) r[e] = relu ? fmaxf(c4[e], 0.f) : c4[e];
    if (skip) {
        const uint2 sk = *reinterpret_cast<const uint2 *>(skip + o);
        r[0] += bf2f(static_cast<uint16_t>(sk.x & 0xFFFFu));
        r[1] += bf2f(static_cast<uint16_t>(sk.x >> 16));
        r[2] += bf2f(static_cast<uint16_t>(sk.y & 0xFFFFu));
        r[3] += bf2f(static_cast<uint16_t>(sk.y >> 16));
    }
    *reinterpret_cast<uint2 *>(out + o) = uint2{pack2(r[0], r[1]), pack2(r[2], r[3])};
}

// ---------------------------------------------------------------- forward
// out[v][co] = act(b[co] + sum_t sum_ci in[v + off_t][ci] * W[t][ci][co]) (+ skip[v][co])
// Wt is [27][COUT][CIN].  UP: the input lives at half resolution and is read
// nearest-upsampled.  pre (optional): the pre-activation values.
//
// UP is evaluated on the coarse input directly: along each axis a fine
// voxel of parity p reads coarse offsets floor((p + d) / 2) for its taps
// d = -1, 0, 1, which are p - 1 and p, and a tap outside the fine volume is
// exactly a coarse offset outside the coarse one.  So the 27-tap
// convolution of the upsampled input equals, per parity (px, py, pz), a
// 2x2x2 convolution of the coarse input with the weights of the fine taps
// that meet on each coarse tap summed (weights_up_bf16: Wt is then
// [8 parities][8 taps][COUT][CIN]).  A wavefront's voxel tiles each hold 16
// voxels of one x parity (every other voxel), so the weight operand is the
// same for all columns of a tile and the tile reads 16 consecutive coarse
// voxels; y and z parities are those of the wavefront's row and plane.
//
// An implicit GEMM D[co][v] += sum_k A[co][k] B[k][v] over k = (tap, ci) on
// v_mfma_f32_16x16x32_bf16.  A wavefront owns one row of NV x 16 consecutive
// voxels along x and all COUT / 16 output-channel tiles, so per K step of 32
// it loads COUT / 16 weight operands and NV input operands (16 bytes per
// lane each, contiguous in the channel) and issues (COUT / 16) x NV matrix
// instructions on them.  A K step is 32 channels of one tap (CIN >= 32) or
// 16 channels of two consecutive taps (CIN = 16, the 28th tap reads zero).
// Operand layouts (both operands give lane l the same eight k, so their
// order within the lane does not change the sum):
//   A (16x32): lane l holds row l%16, k = 8*(l/16) .. +7
//   B (32x16): lane l holds column l%16, k = 8*(l/16) .. +7
//   D (16x16 FP32): lane l holds D[4*(l/16) .. +3][l%16]
// The epilogue stores the four channels a lane holds as one 8-byte write.
//
// GRAD: the data gradient of a convolution that is not upsampled, the same
// GEMM with mirrored taps: in is the output's gradient (BF16), CIN the
// layer's output and COUT its input channels, Wt its weights as
// [27][COUT][CIN] ([tap][c_in][c_out] of the layer), and gin receives FP32
// sums, zero where the BF16 activation `skip` (optional) is not positive.
template <int CIN, int COUT, bool UP, int NV, bool GRAD = false>
__global__ void __launch_bounds__(256) k_conv_fwd(Dims D, const uint16_t *__restrict__ in,
                                                  const uint16_t *__restrict__ Wt, const float *__restrict__ bias,
                                                  uint16_t *__restrict__ out, uint16_t *__restrict__ pre,
                                                  const uint16_t *__restrict__ skip, int relu,
                                                  float *__restrict__ gin) {
    static_assert(CIN % 16 == 0 && COUT % 16 == 0, "channels come in tiles of 16");
    static_assert(!(GRAD && UP), "k_conv_up_dgrad is the upsampling layers' data gradient");
    static_assert(!UP || (CIN >= 32 && NV % 2 == 0), "the upsampling form takes 32-channel K steps, tile pairs");
    constexpr int MT = COUT / 16;
    constexpr int KSTEPS = UP ? 8 * (CIN / 32) : (CIN >= 32 ? 27 * (CIN / 32) : 14);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int y = static_cast<int>(blockIdx.y) * 4 + wave, z = blockIdx.z;
    const int x0 = static_cast<int>(blockIdx.x) * (16 * NV);
    if (y >= D.Y) return;  // no workgroup barrier in this kernel
    const int col = lane & 15, kg = lane >> 4;
    const Dims C{D.X >> 1, D.Y >> 1, D.Z >> 1};
    const bf16x8 zero8 = __builtin_bit_cast(bf16x8, uint4{0u, 0u, 0u, 0u});
    f32x4 acc[MT][NV];
#pragma unroll
    for (int ct = 0; ct < MT; ct++)
#pragma unroll
        for (int j = 0; j < NV; j++) acc[ct][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (UP) {
        const int py = y & 1, pz = z & 1;
        for (int st = 0; st < KSTEPS; st++) {
            const int t8 = st / (CIN / 32), c = (st % (CIN / 32)) * 32 + 8 * kg;
            const int ox = t8 & 1, oy = (t8 >> 1) & 1, oz = t8 >> 2;
            bf16x8 a[2][MT], b[NV];
#pragma unroll
            for (int px = 0; px < 2; px++)
#pragma unroll
                for (int ct = 0; ct < MT; ct++)
                    a[px][ct] = __builtin_bit_cast(
                        bf16x8, *reinterpret_cast<const uint4 *>(
                                    Wt + ((static_cast<long long>(((pz * 2 + py) * 2 + px) * 8 + t8)) * COUT + ct * 16 +
                                          col) * CIN + c));
            const int cy = (y >> 1) + py - 1 + oy, cz = (z >> 1) + pz - 1 + oz;
            const bool row_ok = cy >= 0 && cy < C.Y && cz >= 0 && cz < C.Z;
#pragma unroll
            for (int j = 0; j < NV; j++) {
                const int cx = x0 / 2 + 16 * (j / 2) + col + (j & 1) - 1 + ox;
                b[j] = zero8;
                if (row_ok && cx >= 0 && cx < C.X)
                    b[j] = __builtin_bit_cast(bf16x8,
                                              *reinterpret_cast<const uint4 *>(in + vox(C, cx, cy, cz) * CIN + c));
            }
#pragma unroll
            for (int ct = 0; ct < MT; ct++)
#pragma unroll
                for (int j = 0; j < NV; j++)
                    acc[ct][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[j & 1][ct], b[j], acc[ct][j], 0, 0, 0);
        }
    }
    for (int st = 0; st < (UP ? 0 : KSTEPS); st++) {
        // tap and first channel of this lane's eight k values
        int t, c;
        if (CIN >= 32) {
            t = st / (CIN / 32);
            c = (st % (CIN / 32)) * 32 + 8 * kg;
        } else {
            t = 2 * st + (kg >> 1);
            c = 8 * (kg & 1);
        }
        const bool tap_ok = t < 27;
        int dx, dy, dz;
        tap_offset(tap_ok ? t : 0, dx, dy, dz);
        if (GRAD) {
            dx = -dx;
            dy = -dy;
            dz = -dz;
        }
        bf16x8 a[MT], b[NV];
#pragma unroll
        for (int ct = 0; ct < MT; ct++)
            a[ct] = tap_ok ? __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4 *>(
                                                            Wt + (static_cast<long long>(t) * COUT + ct * 16 + col) *
                                                                     CIN + c))
                           : zero8;
        const int yy = y + dy, zz = z + dz;
        const bool row_ok = tap_ok && yy >= 0 && yy < D.Y && zz >= 0 && zz < D.Z;
#pragma unroll
        for (int j = 0; j < NV; j++) {
            const int xx = x0 + 16 * j + col + dx;
            b[j] = zero8;
            if (row_ok && xx >= 0 && xx < D.X)
                b[j] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4 *>(in + vox(D, xx, yy, zz) * CIN + c));
        }
#pragma unroll
        for (int ct = 0; ct < MT; ct++)
#pragma unroll
            for (int j = 0; j < NV; j++)
                acc[ct][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[ct], b[j], acc[ct][j], 0, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < NV; j++) {
        const int vx = UP ? x0 + 32 * (j / 2) + 2 * col + (j & 1) : x0 + 16 * j + col;
        if (vx >= D.X) continue;
        const long long v = vox(D, vx, y, z);
#pragma unroll
        for (int ct = 0; ct < MT; ct++) {
            const int co = ct * 16 + 4 * kg;
            store_tile<GRAD>(acc[ct][j], bias + co, v * COUT + co, out, pre, skip, relu, gin);
        }
    }
}

// ---- the two 16-channel layers at full resolution
// With 16 output channels every 16-byte load of k_conv_fwd feeds one matrix
// instruction, and each input row is loaded for all 27 taps: at 256x128x128
// these layers were bound by the L1 (64 bytes per clock and CU: 165 and 199
// us), three times over what memory needs.  Both kernels march along z with
// the sums of the output planes an input plane reaches in registers, so a
// row is loaded once per shift along x and wavefront.  A row is read through
// a buffer descriptor of its own: voxels beyond its ends read as zero.
__device__ __forceinline__ bf16x8 row_load(__amdgpu_buffer_rsrc_t r, unsigned offset) {
    return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(r, offset, 0, 0));
}
// row (y, z) of a volume of C channels (outside the volume: empty)
template <int C>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t row_buffer(const Dims &D, const uint16_t *in, int y, int z) {
    const bool ok = y >= 0 && y < D.Y && z >= 0 && z < D.Z;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(in + (ok ? vox(D, 0, y, z) * C : 0)),
                                             static_cast<short>(0), ok ? D.X * 2 * C : 0, 0x00020000);
}
constexpr unsigned kNowhere = 0x80000000u;  // an offset beyond any row

// 16 -> 16 channels at one resolution (k_conv_fwd's arguments).  A wavefront
// owns 16 voxels along x and kRows16 rows, with the weights of all taps in
// registers: per row of taps one operand for the voxels x - 1 and x, one for
// x + 1 (its other half zero).  At 256x128x128 165 -> 88 us (57 to read and
// write the volume once), its gradient form at 128x64x64 30 -> 21 us; loading
// the next plane ahead takes the second wavefront per SIMD (130 us).
constexpr int kRows16 = 4;
template <bool GRAD>
__global__ void __launch_bounds__(256) k_conv16(Dims D, const uint16_t *__restrict__ in, const uint16_t *__restrict__ Wt,
                                                const float *__restrict__ bias, uint16_t *__restrict__ out,
                                                uint16_t *__restrict__ pre, const uint16_t *__restrict__ skip, int relu,
                                                float *__restrict__ gin, int planes) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    const int col = lane & 15, kg = lane >> 4;
    const int x0 = static_cast<int>(blockIdx.x) * 16, y0 = (static_cast<int>(blockIdx.y) * 4 + wave) * kRows16;
    const int z0 = static_cast<int>(blockIdx.z) * planes, z1 = min(z0 + planes, D.Z);
    if (y0 >= D.Y) return;  // no workgroup barrier in this kernel
    const bf16x8 zero8 = __builtin_bit_cast(bf16x8, uint4{0u, 0u, 0u, 0u});
    bf16x8 a[9][2];  // [3 (dz + 1) + dy + 1 of the input row][voxels x - 1 and x; x + 1]
#pragma unroll
    for (int r = 0; r < 9; r++)
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const int d = q == 0 ? kg >> 1 : 2;
            const int t = GRAD ? (8 - r) * 3 + 2 - d : r * 3 + d;
            const bf16x8 w =
                __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4 *>(Wt + (t * 16 + col) * 16 + 8 * (kg & 1)));
            a[r][q] = q == 1 && kg >= 2 ? zero8 : w;
        }
    const int left = (x0 + col - 1) * 32 + 16 * kg;
    const unsigned off0 = left < 0 ? kNowhere : static_cast<unsigned>(left);
    const unsigned off1 = kg >= 2 ? kNowhere : static_cast<unsigned>((x0 + col + 1) * 32 + 16 * kg);
    f32x4 acc[3][kRows16];
    // input plane z0 - 1 + q, q % 3 == PH: starts output plane z0 + q (slot
    // PH), ends z0 + q - 2 (slot PH + 1 mod 3)
    auto plane = [&](auto ph, int q) {
        constexpr int PH = decltype(ph)::value;
        const int zi = z0 - 1 + q;
#pragma unroll
        for (int o = 0; o < kRows16; o++) acc[PH][o] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (zi >= 0 && zi < D.Z) {
            bf16x8 b[kRows16 + 2][2];
#pragma unroll
            for (int r = 0; r < kRows16 + 2; r++) {
                const auto buf = row_buffer<16>(D, in, y0 - 1 + r, zi);
                b[r][0] = row_load(buf, off0);
                b[r][1] = row_load(buf, off1);
            }
#pragma unroll
            for (int r = 0; r < kRows16 + 2; r++)
#pragma unroll
                for (int h = 0; h < 2; h++)
#pragma unroll
                    for (int dz = 0; dz < 3; dz++)
#pragma unroll
                        for (int dy = 0; dy < 3; dy++) {
                            const int o = r - dy;
                            if (o < 0 || o >= kRows16) continue;
                            f32x4 &c = acc[(PH + 3 - dz) % 3][o];
                            c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[3 * dz + dy][h], b[r][h], c, 0, 0, 0);
                        }
        }
        const int z = zi - 1;
        if (z < z0 || z >= z1 || x0 + col >= D.X) return;
#pragma unroll
        for (int o = 0; o < kRows16; o++)
            if (y0 + o < D.Y)
                store_tile<GRAD>(acc[(PH + 1) % 3][o], bias + 4 * kg, vox(D, x0 + col, y0 + o, z) * 16 + 4 * kg, out, pre,
                                 skip, relu, gin);
    };
#pragma unroll 1
    for (int q = 0; q < z1 - z0 + 2; q += 3) {
        plane(std::integral_constant<int, 0>(), q);
        if (q + 1 < z1 - z0 + 2) plane(std::integral_constant<int, 1>(), q + 1);
        if (q + 2 < z1 - z0 + 2) plane(std::integral_constant<int, 2>(), q + 2);
    }
}

// 32 -> 16 channels, the input upsampled (k_conv_fwd's UP form).  A wavefront
// owns 16 coarse voxels along x and two coarse rows, that is 2 x 2 parities
// of four fine rows, and marches through the coarse planes: plane c ends the
// fine planes 2 c - 1 and 2 c and starts 2 c + 1 and 2 c + 2.  The 64 weight
// operands lie in LDS, each read once per plane for two rows.  At 256x128x128
// 199 -> 170 us, with two wavefronts per SIMD to hide the loads (64 us of
// memory); the next plane ahead needs more registers than two leave (259 us).
__global__ void __launch_bounds__(256) k_conv_up16(Dims D, const uint16_t *__restrict__ in,
                                                   const uint16_t *__restrict__ Wt, const float *__restrict__ bias,
                                                   uint16_t *__restrict__ out, uint16_t *__restrict__ pre,
                                                   const uint16_t *__restrict__ skip, int relu, int planes) {
    __shared__ uint4 weights[64][64];  // [parity][tap], as a lane reads it
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    const int col = lane & 15, kg = lane >> 4;
    const Dims C{D.X >> 1, D.Y >> 1, D.Z >> 1};
    for (int m = wave; m < 64; m += 4)
        weights[m][lane] = *reinterpret_cast<const uint4 *>(Wt + (m * 16 + col) * 32 + 8 * kg);
    __syncthreads();
    const int x0 = static_cast<int>(blockIdx.x) * 16, y0 = (static_cast<int>(blockIdx.y) * 4 + wave) * 2;
    const int c0 = static_cast<int>(blockIdx.z) * planes, c1 = min(c0 + planes, C.Z);
    if (y0 >= C.Y) return;  // no workgroup barrier from here on
    unsigned off[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const int o = (x0 + col - 1 + d) * 64 + 16 * kg;
        off[d] = o < 0 ? kNowhere : static_cast<unsigned>(o);
    }
    f32x4 acc[2][2][2][2][2];  // [pair of fine planes, by parity of c][odd plane first][coarse row][y parity][x parity]
    auto plane = [&](auto ph, int c) {
        constexpr int END = decltype(ph)::value, BEGIN = 1 - END;
#pragma unroll
        for (int n = 0; n < 16; n++)
            acc[BEGIN][n >> 3][(n >> 2) & 1][(n >> 1) & 1][n & 1] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (c >= 0 && c < C.Z) {
            bf16x8 b[4][3];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const auto buf = row_buffer<32>(C, in, y0 - 1 + r, c);
#pragma unroll
                for (int d = 0; d < 3; d++) b[r][d] = row_load(buf, off[d]);
            }
#pragma unroll
            for (int m = 0; m < 64; m++) {
                const int px = (m >> 3) & 1, py = (m >> 4) & 1, pz = m >> 5, ox = m & 1, oy = (m >> 1) & 1, oz = (m >> 2) & 1;
                const bf16x8 w = __builtin_bit_cast(bf16x8, weights[m][lane]);
#pragma unroll
                for (int r = 0; r < 2; r++) {
                    f32x4 &s = acc[oz == 1 ? END : BEGIN][1 - pz][r][py][px];
                    s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, b[r + py + oy][px + ox], s, 0, 0, 0);
                }
            }
        }
#pragma unroll
        for (int n = 0; n < 16; n++) {
            const int even = n >> 3, r = (n >> 2) & 1, py = (n >> 1) & 1, px = n & 1;
            const int z = 2 * c - 1 + even, y = 2 * (y0 + r) + py, x = 2 * (x0 + col) + px;
            if (z >= 2 * c0 && z < 2 * c1 && y < D.Y && x < D.X)
                store_tile<false>(acc[END][even][r][py][px], bias + 4 * kg, vox(D, x, y, z) * 16 + 4 * kg, out, pre, skip,
                                  relu, nullptr);
        }
    };
#pragma unroll
    for (int n = 0; n < 16; n++) acc[0][n >> 3][(n >> 2) & 1][(n >> 1) & 1][n & 1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int c = c0 - 1; c <= c1; c += 2) {
        plane(std::integral_constant<int, 0>(), c);
        if (c + 1 <= c1) plane(std::integral_constant<int, 1>(), c + 1);
    }
}

// First layer: two FP32 channels to 16 BF16 with ReLU, on
// v_mfma_f32_16x16x4_f32 (FP32 operands and sums) in the manner of k_conv16:
// a K step is two voxels of two channels.  A row of three taps is one step
// for the voxels x - 1 and x; the voxels x + 1 of two rows share one, so a
// plane of taps is five steps.  One thread per voxel with 864 multiply-adds was
// bound by their issue: 169 us at 256x128x128, 106 now (58 of matrix issue).
__global__ void __launch_bounds__(256) k_conv_in(Dims D, const float *__restrict__ x, const float *__restrict__ W,
                                                 const float *__restrict__ bias, uint16_t *__restrict__ out,
                                                 int planes) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    const int col = lane & 15, kg = lane >> 4;
    const int x0 = static_cast<int>(blockIdx.x) * 16, y0 = (static_cast<int>(blockIdx.y) * 4 + wave) * kRows16;
    const int z0 = static_cast<int>(blockIdx.z) * planes, z1 = min(z0 + planes, D.Z);
    if (y0 >= D.Y) return;  // no workgroup barrier in this kernel
    auto weight = [&](int t, int ci) { return W[(t * 2 + ci) * 16 + col]; };
    float a[3][5];  // [dz + 1][rows dy = -1, 0, 1 at x - 1 and x; x + 1 of rows -1 and 0; x + 1 of row 1]
#pragma unroll
    for (int dz = 0; dz < 3; dz++) {
#pragma unroll
        for (int dy = 0; dy < 3; dy++) a[dz][dy] = weight((dz * 3 + dy) * 3 + (kg >> 1), kg & 1);
        a[dz][3] = weight((dz * 3 + (kg >> 1)) * 3 + 2, kg & 1);
        a[dz][4] = kg < 2 ? weight((dz * 3 + 2) * 3 + 2, kg & 1) : 0.f;
    }
    const int left = (x0 + col - 1) * 8 + 4 * kg;
    const unsigned off0 = left < 0 ? kNowhere : static_cast<unsigned>(left);
    const unsigned right = static_cast<unsigned>((x0 + col + 1) * 8 + 4 * (kg & 1));
    const unsigned off_lo = kg < 2 ? right : kNowhere, off_hi = kg < 2 ? kNowhere : right;
    f32x4 acc[3][kRows16];
    auto plane = [&](auto ph, int q) {
        constexpr int PH = decltype(ph)::value;
        const int zi = z0 - 1 + q;
#pragma unroll
        for (int o = 0; o < kRows16; o++) acc[PH][o] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (zi >= 0 && zi < D.Z) {
            unsigned b0[kRows16 + 2], lo[kRows16 + 2], hi[kRows16 + 2];
#pragma unroll
            for (int r = 0; r < kRows16 + 2; r++) {
                const int y = y0 - 1 + r;
                const bool ok = y >= 0 && y < D.Y;
                const auto buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(x + (ok ? vox(D, 0, y, zi) * 2 : 0)),
                                                                   static_cast<short>(0), ok ? D.X * 8 : 0, 0x00020000);
                b0[r] = __builtin_amdgcn_raw_buffer_load_b32(buf, off0, 0, 0);
                lo[r] = __builtin_amdgcn_raw_buffer_load_b32(buf, off_lo, 0, 0);
                hi[r] = r >= 1 && r <= kRows16 ? __builtin_amdgcn_raw_buffer_load_b32(buf, off_hi, 0, 0) : 0u;
            }
#pragma unroll
            for (int o = 0; o < kRows16; o++)
#pragma unroll
                for (int dz = 0; dz < 3; dz++) {
                    f32x4 &c = acc[(PH + 3 - dz) % 3][o];
#pragma unroll
                    for (int dy = 0; dy < 3; dy++)
                        c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[dz][dy], __uint_as_float(b0[o + dy]), c, 0, 0, 0);
                    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[dz][3], __uint_as_float(lo[o] | hi[o + 1]), c, 0, 0, 0);
                    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[dz][4], __uint_as_float(lo[o + 2]), c, 0, 0, 0);
                }
        }
        const int z = zi - 1;
        if (z < z0 || z >= z1 || x0 + col >= D.X) return;
#pragma unroll
        for (int o = 0; o < kRows16; o++)
            if (y0 + o < D.Y)
                store_tile<false>(acc[(PH + 1) % 3][o], bias + 4 * kg, vox(D, x0 + col, y0 + o, z) * 16 + 4 * kg, out,
                                  nullptr, nullptr, 1, nullptr);
    };
#pragma unroll 1
    for (int q = 0; q < z1 - z0 + 2; q += 3) {
        plane(std::integral_constant<int, 0>(), q);
        if (q + 1 < z1 - z0 + 2) plane(std::integral_constant<int, 1>(), q + 1);
        if (q + 2 < z1 - z0 + 2) plane(std::integral_constant<int, 2>(), q + 2);
    }
}

// Last layer: CI BF16 channels -> one FP32 output, no activation.  A thread
// owns NZ voxels of one (x, y) column and marches through the input planes
// z0-1 .. z0+NZ: each tap value it loads (16 bytes per eight channels) is
// added, with the weight of its z offset, to each of the up to three
// outputs whose stencil holds that plane.  Every output still receives its
// terms in tap order (z offset, then y, x, channel), skipping taps outside
// the volume, as a per-voxel loop over the 27 taps adds them.
template <int CI, int NZ>
__global__ void k_conv_out(Dims D, const uint16_t *__restrict__ in, const float *__restrict__ W,
                           const float *__restrict__ bias, float *__restrict__ y) {
    static_assert(CI % 8 == 0, "channels in groups of eight");
    const int i = static_cast<int>(blockIdx.x) * 64 + static_cast<int>(threadIdx.x);
    const int j = static_cast<int>(blockIdx.y) * 4 + static_cast<int>(threadIdx.y);
    const int z0 = static_cast<int>(blockIdx.z) * NZ;
    if (i >= D.X || j >= D.Y) return;
    float acc[NZ];
#pragma unroll
    for (int q = 0; q < NZ; q++) acc[q] = bias[0];
#pragma unroll
    for (int r = 0; r < NZ + 2; r++) {
        const int zp = z0 - 1 + r;  // input plane; feeds outputs q = r (dz -1), r - 1 (dz 0), r - 2 (dz +1)
        if (zp < 0 || zp >= D.Z) continue;
#pragma unroll
        for (int dy = -1; dy <= 1; dy++) {
            const int yy = j + dy;
            if (yy < 0 || yy >= D.Y) continue;
#pragma unroll
            for (int dx = -1; dx <= 1; dx++) {
                const int xx = i + dx;
                if (xx < 0 || xx >= D.X) continue;
                const uint4 *src = reinterpret_cast<const uint4 *>(in + vox(D, xx, yy, zp) * CI);
                const int tb = (dy + 1) * 3 + (dx + 1);  // tap within its z plane
#pragma unroll
                for (int g = 0; g < CI / 8; g++) {
                    const uint4 qv = src[g];
                    const unsigned w4[4] = {qv.x, qv.y, qv.z, qv.w};
#pragma unroll
                    for (int e = 0; e < 8; e++) {
                        const float v = bf2f(static_cast<uint16_t>((w4[e >> 1] >> (16 * (e & 1))) & 0xFFFFu));
                        const int ci = 8 * g + e;
                        if (r < NZ) acc[r] = fmaf(v, W[tb * CI + ci], acc[r]);
                        if (r >= 1 && r - 1 < NZ) acc[r - 1] = fmaf(v, W[(9 + tb) * CI + ci], acc[r - 1]);
                        if (r >= 2) acc[r - 2] = fmaf(v, W[(18 + tb) * CI + ci], acc[r - 2]);
                    }
                }
            }
        }
    }
#pragma unroll
    for (int q = 0; q < NZ; q++)
        if (z0 + q < D.Z) y[vox(D, i, j, z0 + q)] = acc[q];
}

// 2x2x2 mean, D: the output (coarse) dims
template <int C>
__global__ void k_down(Dims D, const uint16_t *__restrict__ in, uint16_t *__restrict__ out) {
    const long long n = static_cast<long long>(D.X) * D.Y * D.Z * C;
    const Dims F{D.X * 2, D.Y * 2, D.Z * 2};
    for (long long q = blockIdx.x * 256LL + threadIdx.x; q < n; q += 256LL * gridDim.x) {
        const int c = static_cast<int>(q % C);
        const long long v = q / C;
        const int x = static_cast<int>(v % D.X), y = static_cast<int>((v / D.X) % D.Y),
                  z = static_cast<int>(v / (static_cast<long long>(D.X) * D.Y));
        float s = 0.f;
        for (int o = 0; o < 8; o++) s += bf2f(in[vox(F, 2 * x + (o & 1), 2 * y + ((o >> 1) & 1), 2 * z + (o >> 2)) * C + c]);
        out[q] = f2bf(s * 0.125f);
    }
}

// ---------------------------------------------------------------- backward
// One 64-bit transposed LDS read per lane: with the 16 lanes of a group
// pointing at four voxels (lane 4 i + q at channels 4 q .. 4 q + 3 of voxel
// i), lane c of the group receives channel c of the four voxels.
__device__ inline bf16x4 lds_transposed(const uint16_t *p) {
    typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;
    return __builtin_bit_cast(
        bf16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_bf16x4 *)(const_cast<uint16_t *>(p))));
}
__device__ inline bf16x8 join(bf16x4 a, bf16x4 b) {
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

// Weight gradient of a 3x3x3 convolution, partial sums:
// part[block][t][ci][co] = sum over the block's voxels v of
// in[v + off_t][ci] * g[v][co], both BF16, FP32 accumulation.
//
// A matrix product over the voxels: A is in^T (rows ci), B is g (columns co),
// K = 32 voxels per instruction.  A workgroup covers the nine taps of one z
// offset (blockIdx.y), one wavefront per y offset with the three x offsets in
// its registers.  It stages rows of g and of `in` with a one-voxel halo in
// LDS as they lie in memory, [voxel][channel] (zero outside the volume), and
// reads operands with the transposing LDS read: a tap is only another base
// address, and an operand of g serves three taps.  Voxels are padded to an
// odd multiple of 32 bytes where they are 64 bytes or more, so that the eight
// voxels a read touches at once lie in different banks.  UP: `in` lives at
// half resolution; a fine voxel's operand address is that of its coarse voxel.
//
// With two-byte gathers from memory and one atomic per weight and wavefront
// the layers of a 128x64x64 volume took 1400 us together; so they take 185 us.
constexpr int kGradVoxels = 256;  // voxels per staged block (about), multiple of 32
constexpr int kGradSegment = 128; // longest x segment of a block
template <int C>
constexpr int lds_voxel() {
    return C == 16 ? 16 : C + 16;  // uint16 per voxel
}
struct GradBlocks {
    int xb, rows;        // voxels along x and rows along y of a block
    int nx, ny, blocks;  // blocks along x and y, in all
};
inline GradBlocks grad_blocks(Dims D) {
    GradBlocks b;
    b.xb = D.X < kGradSegment ? D.X : kGradSegment;
    int rows = kGradVoxels / b.xb;
    rows = rows < 2 ? 2 : (rows > 64 ? 64 : rows & ~1);
    const int even = (D.Y + 1) & ~1;
    b.rows = rows < even ? rows : even;
    b.nx = (D.X + b.xb - 1) / b.xb;
    b.ny = (D.Y + b.rows - 1) / b.rows;
    b.blocks = b.nx * b.ny * D.Z;
    return b;
}
template <int CIN, int COUT, bool UP>
__global__ void __launch_bounds__(192) k_conv_wgrad(Dims D, GradBlocks B, const uint16_t *__restrict__ in,
                                                    const uint16_t *__restrict__ g, float *__restrict__ part) {
    constexpr int GS = lds_voxel<COUT>(), IS = lds_voxel<CIN>(), MT = CIN / 16, NT = COUT / 16;
    extern __shared__ __align__(16) uint16_t lds[];
    const int fmax = (B.rows * B.xb + 31) & ~31;
    const int rows_in = UP ? B.rows / 2 + 2 : B.rows + 2, xh = UP ? (B.xb + 1) / 2 + 2 : B.xb + 2;
    uint16_t *sg = lds, *si = sg + fmax * GS;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int dz = static_cast<int>(blockIdx.y) - 1, dy = wave - 1;
    const Dims C{UP ? D.X >> 1 : D.X, UP ? D.Y >> 1 : D.Y, UP ? D.Z >> 1 : D.Z};
    f32x4 acc[3][MT][NT];
#pragma unroll
    for (int d = 0; d < 3; d++)
#pragma unroll
        for (int a = 0; a < MT; a++)
#pragma unroll
            for (int b = 0; b < NT; b++) acc[d][a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    // the voxels (of 32 in a K step) whose chunk this lane's two reads fetch
    const int k0 = 4 * (lane >> 4) + ((lane & 15) >> 2), q4 = 4 * (lane & 3);
    for (int blk = blockIdx.x; blk < B.blocks; blk += gridDim.x) {
        const int bx = blk % B.nx, by = (blk / B.nx) % B.ny, z = blk / (B.nx * B.ny);
        if (z + dz < 0 || z + dz >= D.Z) continue;  // uniform over the workgroup
        const int x0 = bx * B.xb, y0 = by * B.rows, zi = UP ? (z + dz) >> 1 : z + dz;
        const int cx0 = UP ? (x0 >> 1) - 1 : x0 - 1, cy0 = UP ? (y0 >> 1) - 1 : y0 - 1;
        for (unsigned q = threadIdx.x; q < static_cast<unsigned>(fmax * (COUT / 8)); q += 192) {
            const unsigned f = q / (COUT / 8), c = q % (COUT / 8) * 8, r = f / B.xb;
            const int x = x0 + static_cast<int>(f - r * B.xb), y = y0 + static_cast<int>(r);
            uint4 v{0u, 0u, 0u, 0u};
            if (static_cast<int>(r) < B.rows && x < D.X && y < D.Y)
                v = *reinterpret_cast<const uint4 *>(g + vox(D, x, y, z) * COUT + c);
            *reinterpret_cast<uint4 *>(sg + f * GS + c) = v;
        }
        for (unsigned q = threadIdx.x; q < static_cast<unsigned>(rows_in * xh * (CIN / 8)); q += 192) {
            const unsigned p = q / (CIN / 8), c = q % (CIN / 8) * 8, r = p / xh;
            const int x = cx0 + static_cast<int>(p - r * xh), y = cy0 + static_cast<int>(r);
            uint4 v{0u, 0u, 0u, 0u};
            if (x >= 0 && x < C.X && y >= 0 && y < C.Y)
                v = *reinterpret_cast<const uint4 *>(in + vox(C, x, y, zi) * CIN + c);
            *reinterpret_cast<uint4 *>(si + p * IS + c) = v;
        }
        __syncthreads();
        for (int f0 = 0; f0 < fmax; f0 += 32) {
            bf16x4 gb[2][NT], ia[2][3][MT];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int f = f0 + k0 + 16 * h;
#pragma unroll
                for (int b = 0; b < NT; b++) gb[h][b] = lds_transposed(sg + f * GS + b * 16 + q4);
                // positions past the block's last row (g is zero there) read the last row
                const int r0 = f / B.xb, x = f - r0 * B.xb, r = r0 < B.rows ? r0 : B.rows - 1;
#pragma unroll
                for (int d = 0; d < 3; d++) {
                    const int px = UP ? ((x0 + x + d - 1) >> 1) - cx0 : x + d,
                              py = UP ? ((y0 + r + dy) >> 1) - cy0 : r + dy + 1;
#pragma unroll
                    for (int a = 0; a < MT; a++) ia[h][d][a] = lds_transposed(si + (py * xh + px) * IS + a * 16 + q4);
                }
            }
#pragma unroll
            for (int d = 0; d < 3; d++)
#pragma unroll
                for (int a = 0; a < MT; a++)
#pragma unroll
                    for (int b = 0; b < NT; b++)
                        acc[d][a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            join(ia[0][d][a], ia[1][d][a]), join(gb[0][b], gb[1][b]), acc[d][a][b], 0, 0, 0);
        }
        __syncthreads();
    }
    float *row = part + static_cast<size_t>(blockIdx.x) * (27 * CIN * COUT);
#pragma unroll
    for (int d = 0; d < 3; d++)
#pragma unroll
        for (int a = 0; a < MT; a++)
#pragma unroll
            for (int b = 0; b < NT; b++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int t = (dz + 1) * 9 + (dy + 1) * 3 + d, ci = a * 16 + 4 * (lane >> 4) + e,
                              co = b * 16 + (lane & 15);
                    row[(t * CIN + ci) * COUT + co] = acc[d][a][b][e];
                }
}

// the workgroup's sum of one float4 per thread over the threads with the same
// threadIdx.x % groups (a power of two up to 16), written by the first
// `groups` threads to row[4 * group ..]; 256 threads
__device__ inline void group_sums(float4 v, int groups, float *row) {
    __shared__ float4 s[256];
    s[threadIdx.x] = v;
    __syncthreads();
    for (int n = 128; n >= groups; n >>= 1) {
        if (static_cast<int>(threadIdx.x) < n) {
            const float4 a = s[threadIdx.x], b = s[threadIdx.x + n];
            s[threadIdx.x] = float4{a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w};
        }
        __syncthreads();
    }
    if (static_cast<int>(threadIdx.x) < groups) *reinterpret_cast<float4 *>(row + 4 * threadIdx.x) = s[threadIdx.x];
}

// Data gradient of an upsampling layer with the sum over the eight fine
// children of a coarse voxel: gc[c][ci] = sum over the 4x4x4 fine voxels
// 2 c - 1 .. 2 c + 2 of g[v][co] Wd[tap][ci][co], the transpose of the
// 2x2x2-per-parity form k_conv_fwd evaluates forward.  64 taps instead of the
// 27 x 8 of a fine-resolution gradient followed by the sum, and that fine
// FP32 gradient (67 MB at 128x64x64) is never written.  A weight Wd is a sum
// of up to eight BF16 weights, held as three BF16 terms (the rounded sum and
// twice the rounded remainder: 24 bits), so that the products are those of
// the 27-tap form and no weight is rounded twice.
//
// The workgroup's WAVES wavefronts share one tile of NV x 16 coarse voxels of
// a row and split the 64 taps; their sums meet in LDS in a fixed order, and the epilogue writes the skip gradient (FP32, optional) and
// the gradient under the mask act > 0 (BF16, the next products' operand), and
// keeps the masked values' channel sums (the bias gradient) per workgroup.
// Small levels have few row tiles: there blockIdx.y splits the input channels
// as well, MT tiles of 16 per workgroup (d2's level of a 128x64x64 volume, 64
// row tiles: 49 us with all four channel tiles in one workgroup, 17 us split).
template <int CO, int CI, int NV, int WAVES, int MT>
__global__ void __launch_bounds__(64 * WAVES) k_conv_up_dgrad(Dims D, const uint16_t *__restrict__ g,
                                                       const uint16_t *__restrict__ Wd,
                                                       const uint16_t *__restrict__ act, float *__restrict__ gskip,
                                                       uint16_t *__restrict__ gmask, float *__restrict__ part) {
    constexpr int TILES = MT * NV, TAPS = 64 / WAVES, STEPS = CO == 16 ? TAPS / 2 : TAPS * (CO / 32);
    static_assert(TAPS >= 4 && TAPS <= 16, "a wavefront's taps lie in one z plane, whole rows of four");
    __shared__ f32x4 sum[WAVES][TILES][64];
    __shared__ float bias[WAVES][16 * MT];
    const int ci0 = static_cast<int>(blockIdx.y) * (16 * MT);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, kg = lane >> 4;
    const Dims F{2 * D.X, 2 * D.Y, 2 * D.Z};
    const int nx = (D.X + 16 * NV - 1) / (16 * NV), tiles = nx * D.Y * D.Z;

    const bf16x8 zero8 = __builtin_bit_cast(bf16x8, uint4{0u, 0u, 0u, 0u});
    float4 bct[MT];
#pragma unroll
    for (int ct = 0; ct < MT; ct++) bct[ct] = float4{0.f, 0.f, 0.f, 0.f};
    for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const int x0 = tile % nx * (16 * NV), y = (tile / nx) % D.Y, z = tile / (nx * D.Y);
        f32x4 acc[MT][NV];
#pragma unroll
        for (int ct = 0; ct < MT; ct++)
#pragma unroll
            for (int j = 0; j < NV; j++) acc[ct][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        const int fz = 2 * z - 1 + wave * TAPS / 16;
        if (fz >= 0 && fz < F.Z) {
#pragma unroll 2
            for (int st = 0; st < STEPS; st++) {
                // tap jx + 4 jy + 16 jz and first channel of the lane's eight k values
                const int t = wave * TAPS + (CO == 16 ? 2 * st + (kg >> 1) : st / (CO / 32));
                const int c = CO == 16 ? 8 * (kg & 1) : st % (CO / 32) * 32 + 8 * kg;
                const int fy = 2 * y - 1 + ((t >> 2) & 3);
                const bool row_ok = fy >= 0 && fy < F.Y;
                bf16x8 a[3][MT], b[NV];
#pragma unroll
                for (int h = 0; h < 3; h++)
#pragma unroll
                    for (int ct = 0; ct < MT; ct++)
                        a[h][ct] = __builtin_bit_cast(
                            bf16x8, *reinterpret_cast<const uint4 *>(
                                        Wd + ((64 * h + t) * CI + ci0 + ct * 16 + col) * CO + c));
#pragma unroll
                for (int j = 0; j < NV; j++) {
                    const int fx = 2 * (x0 + 16 * j + col) - 1 + (t & 3);
                    b[j] = zero8;
                    if (row_ok && fx >= 0 && fx < F.X)
                        b[j] = __builtin_bit_cast(bf16x8,
                                                  *reinterpret_cast<const uint4 *>(g + vox(F, fx, fy, fz) * CO + c));
                }
#pragma unroll
                for (int h = 0; h < 3; h++)
#pragma unroll
                    for (int ct = 0; ct < MT; ct++)
#pragma unroll
                        for (int j = 0; j < NV; j++)
                            acc[ct][j] =
                                __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[h][ct], b[j], acc[ct][j], 0, 0, 0);
            }
        }
#pragma unroll
        for (int ct = 0; ct < MT; ct++)
#pragma unroll
            for (int j = 0; j < NV; j++) sum[wave][ct * NV + j][lane] = acc[ct][j];
        __syncthreads();
#pragma unroll
        for (int q = 0; q < TILES; q += WAVES) {
            const int w = q + wave;
            if (w >= TILES) continue;
            const int ct = w / NV, j = w % NV, vx = x0 + 16 * j + col, ci = ci0 + ct * 16 + 4 * kg;
            if (vx >= D.X) continue;
            f32x4 v = sum[0][w][lane];
#pragma unroll
            for (int p = 1; p < WAVES; p++) v += sum[p][w][lane];
            const long long at = vox(D, vx, y, z) * CI + ci;
            if (gskip) *reinterpret_cast<float4 *>(gskip + at) = float4{v[0], v[1], v[2], v[3]};
            const uint2 m = *reinterpret_cast<const uint2 *>(act + at);
            float4 k;
            k.x = positive(m.x & 0xFFFFu) ? v[0] : 0.f;
            k.y = positive(m.x >> 16) ? v[1] : 0.f;
            k.z = positive(m.y & 0xFFFFu) ? v[2] : 0.f;
            k.w = positive(m.y >> 16) ? v[3] : 0.f;
            *reinterpret_cast<uint2 *>(gmask + at) = uint2{pack2(k.x, k.y), pack2(k.z, k.w)};
#pragma unroll
            for (int c2 = 0; c2 < MT; c2++)
                if (c2 == ct) {
                    bct[c2].x += k.x;
                    bct[c2].y += k.y;
                    bct[c2].z += k.z;
                    bct[c2].w += k.w;
                }
        }
        __syncthreads();
    }
    // channel sums: over the 16 columns of a lane group, then the wavefronts
#pragma unroll
    for (int ct = 0; ct < MT; ct++) {
        float v[4] = {bct[ct].x, bct[ct].y, bct[ct].z, bct[ct].w};
#pragma unroll
        for (int e = 0; e < 4; e++) {
            for (int off = 8; off > 0; off >>= 1) v[e] += __shfl_down(v[e], off, 16);
            if (col == 0) bias[wave][ct * 16 + 4 * kg + e] = v[e];
        }
    }
    __syncthreads();
    if (static_cast<int>(threadIdx.x) < 16 * MT) {
        float v = bias[0][threadIdx.x];
        for (int p = 1; p < WAVES; p++) v += bias[p][threadIdx.x];
        part[static_cast<size_t>(blockIdx.x) * CI + ci0 + threadIdx.x] = v;
    }
}

// Gradient at an encoder layer's output: the skip gradient plus the spread
// mean of the coarser level's (gc, at half resolution), under the mask act >
// 0; BF16 operand of the next products and per-workgroup channel sums.
template <int C>
__global__ void __launch_bounds__(256) k_enc_grad(Dims D, const float *__restrict__ gskip,
                                                  const float *__restrict__ gc, const uint16_t *__restrict__ act,
                                                  uint16_t *__restrict__ gmask, float *__restrict__ part) {
    constexpr int G = C / 4;
    const Dims H{D.X >> 1, D.Y >> 1, D.Z >> 1};
    const long long n = static_cast<long long>(D.X) * D.Y * D.Z * G;
    float4 sum{0.f, 0.f, 0.f, 0.f};
    for (long long q = blockIdx.x * 256LL + threadIdx.x; q < n; q += 256LL * gridDim.x) {
        const unsigned v = static_cast<unsigned>(q / G);
        const int c = static_cast<int>(q % G) * 4;
        const unsigned r = v / static_cast<unsigned>(D.X);
        const int x = static_cast<int>(v - r * D.X), y = static_cast<int>(r % D.Y), z = static_cast<int>(r / D.Y);
        const float4 s = *reinterpret_cast<const float4 *>(gskip + q * 4);
        const float4 p = *reinterpret_cast<const float4 *>(gc + vox(H, x >> 1, y >> 1, z >> 1) * C + c);
        const uint2 m = *reinterpret_cast<const uint2 *>(act + q * 4);
        float4 k;
        k.x = positive(m.x & 0xFFFFu) ? s.x + 0.125f * p.x : 0.f;
        k.y = positive(m.x >> 16) ? s.y + 0.125f * p.y : 0.f;
        k.z = positive(m.y & 0xFFFFu) ? s.z + 0.125f * p.z : 0.f;
        k.w = positive(m.y >> 16) ? s.w + 0.125f * p.w : 0.f;
        *reinterpret_cast<uint2 *>(gmask + q * 4) = uint2{pack2(k.x, k.y), pack2(k.z, k.w)};
        sum.x += k.x;
        sum.y += k.y;
        sum.z += k.z;
        sum.w += k.w;
    }
    group_sums(sum, G, part + static_cast<size_t>(blockIdx.x) * C);
}

// Weight gradients of the end layers on the FP32 matrix instruction, four
// voxels per instruction.  A wavefront takes whole x rows; lane l supplies
// voxel l/16 of the four.  NM: row tiles of 16 of the product.
template <int NM>
__device__ inline void store_end_wgrad(f32x4 (&acc)[NM], int rows, float *row) {
    __shared__ f32x4 s[4][NM][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int a = 0; a < NM; a++) s[wave][a][lane] = acc[a];
    __syncthreads();
    for (int a = wave; a < NM; a += 4) {
        f32x4 v = s[0][a][lane];
        for (int p = 1; p < 4; p++) v += s[p][a][lane];
        for (int e = 0; e < 4; e++) {
            const int m = a * 16 + 4 * (lane >> 4) + e;
            if (m < rows) row[m * 16 + (lane & 15)] = v[e];
        }
    }
}
// first layer: rows m = 2 t + ci of x[v + off_t][ci], row 54 ones (the bias
// gradient), columns co of g[v][co].  Thread-per-weight loops over the voxels
// took 1331 us at 128x64x64 (a serial chain of 2048 voxels per thread);
// 46 us so.
constexpr int kInRows = 55;  // 27 taps x 2 channels and the bias
__global__ void __launch_bounds__(256) k_conv_in_wgrad(Dims D, const float *__restrict__ x,
                                                       const float *__restrict__ g, float *__restrict__ part) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, m0 = lane & 15, k = lane >> 4;
    f32x4 acc[4];
    int dx[4], dy[4], dz[4];
#pragma unroll
    for (int a = 0; a < 4; a++) {
        acc[a] = f32x4{0.f, 0.f, 0.f, 0.f};
        tap_offset((a * 16 + m0) / 2 < 27 ? (a * 16 + m0) / 2 : 13, dx[a], dy[a], dz[a]);
    }
    const int lines = D.Y * D.Z;
    for (int line = blockIdx.x * 4 + wave; line < lines; line += 4 * static_cast<int>(gridDim.x)) {
        const int y = line % D.Y, z = line / D.Y;
        const float *src[4];
        bool ok[4];
#pragma unroll
        for (int a = 0; a < 4; a++) {
            const int yy = y + dy[a], zz = z + dz[a];
            ok[a] = a * 16 + m0 < 54 && yy >= 0 && yy < D.Y && zz >= 0 && zz < D.Z;
            src[a] = x + (ok[a] ? vox(D, 0, yy, zz) : 0) * 2 + (m0 & 1);
        }
        const float *gr = g + vox(D, 0, y, z) * 16;
        for (int i = 0; i < D.X; i += 8) {  // sides are multiples of 8
            float b[2], v[2][4];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                b[h] = gr[(i + 4 * h + k) * 16 + m0];
#pragma unroll
                for (int a = 0; a < 4; a++) {
                    const int xx = i + 4 * h + k + dx[a];
                    const bool in = ok[a] && xx >= 0 && xx < D.X;
                    v[h][a] = src[a][in ? 2 * xx : 0];
                    v[h][a] = in ? v[h][a] : 0.f;
                }
                v[h][3] = m0 == 6 ? 1.f : v[h][3];  // row 54
            }
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int a = 0; a < 4; a++)
                    acc[a] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[h][a], b[h], acc[a], 0, 0, 0);
        }
    }
    store_end_wgrad<4>(acc, kInRows, part + static_cast<size_t>(blockIdx.x) * (kInRows * 16));
}
// last layer: rows t of gy[v - off_t], columns ci of in[v][ci] (its BF16
// input, exact in FP32); 996 us as thread-per-weight loops, 34 us so.
__global__ void __launch_bounds__(256) k_conv_out_wgrad(Dims D, const uint16_t *__restrict__ in,
                                                        const float *__restrict__ gy, float *__restrict__ part) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, m0 = lane & 15, k = lane >> 4;
    f32x4 acc[2];
    int dx[2], dy[2], dz[2];
#pragma unroll
    for (int a = 0; a < 2; a++) {
        acc[a] = f32x4{0.f, 0.f, 0.f, 0.f};
        tap_offset(a * 16 + m0 < 27 ? a * 16 + m0 : 13, dx[a], dy[a], dz[a]);
    }
    const int lines = D.Y * D.Z;
    for (int line = blockIdx.x * 4 + wave; line < lines; line += 4 * static_cast<int>(gridDim.x)) {
        const int y = line % D.Y, z = line / D.Y;
        const float *src[2];
        bool ok[2];
#pragma unroll
        for (int a = 0; a < 2; a++) {
            const int yy = y - dy[a], zz = z - dz[a];
            ok[a] = a * 16 + m0 < 27 && yy >= 0 && yy < D.Y && zz >= 0 && zz < D.Z;
            src[a] = gy + (ok[a] ? vox(D, 0, yy, zz) : 0);
        }
        const uint16_t *ir = in + vox(D, 0, y, z) * 16;
        for (int i = 0; i < D.X; i += 8) {
            float b[2], v[2][2];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                b[h] = bf2f(ir[(i + 4 * h + k) * 16 + m0]);
#pragma unroll
                for (int a = 0; a < 2; a++) {
                    const int xx = i + 4 * h + k - dx[a];
                    const bool inside = ok[a] && xx >= 0 && xx < D.X;
                    v[h][a] = src[a][inside ? xx : 0];
                    v[h][a] = inside ? v[h][a] : 0.f;
                }
            }
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int a = 0; a < 2; a++)
                    acc[a] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[h][a], b[h], acc[a], 0, 0, 0);
        }
    }
    store_end_wgrad<2>(acc, 27, part + static_cast<size_t>(blockIdx.x) * (27 * 16));
}

// Data gradient of the last layer, g[v][ci] = sum_t gy[v - off_t] W[t][ci]:
// the skip gradient (FP32), its masked BF16 form and its channel sums.  The
// FP32 matrix instruction with the weights as its rows, held in seven
// registers over the whole launch (as scalar operands of vector
// multiply-adds they were loaded again for every voxel: 31 us at 128x64x64
// before the masked outputs and sums came in, 64 us with them); 21 us so.
template <int CI>
__global__ void __launch_bounds__(256) k_conv_out_dgrad(Dims D, const float *__restrict__ W,
                                                        const float *__restrict__ gy, const uint16_t *__restrict__ act,
                                                        float *__restrict__ gskip, uint16_t *__restrict__ gmask,
                                                        float *__restrict__ part) {
    static_assert(CI == 16, "one row tile");
    constexpr int STEPS = 7;  // 27 taps in steps of four
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, kg = lane >> 4;
    float a[STEPS];
    int dx[STEPS], dy[STEPS], dz[STEPS];
#pragma unroll
    for (int s = 0; s < STEPS; s++) {
        const int t = 4 * s + kg;
        a[s] = t < 27 ? W[t * CI + col] : 0.f;
        tap_offset(t < 27 ? t : 13, dx[s], dy[s], dz[s]);
    }
    float4 sum{0.f, 0.f, 0.f, 0.f};
    const int lines = D.Y * D.Z;
    for (int line = blockIdx.x * 4 + wave; line < lines; line += 4 * static_cast<int>(gridDim.x)) {
        const int y = line % D.Y, z = line / D.Y;
        const float *src[STEPS];
        bool ok[STEPS];
#pragma unroll
        for (int s = 0; s < STEPS; s++) {
            const int yy = y - dy[s], zz = z - dz[s];
            ok[s] = yy >= 0 && yy < D.Y && zz >= 0 && zz < D.Z;
            src[s] = gy + (ok[s] ? vox(D, 0, yy, zz) : 0);
        }
        for (int x0 = 0; x0 < D.X; x0 += 16) {
            f32x4 acc{0.f, 0.f, 0.f, 0.f};
            float b[STEPS];
#pragma unroll
            for (int s = 0; s < STEPS; s++) {
                const int xx = x0 + col - dx[s];
                const bool inside = ok[s] && xx >= 0 && xx < D.X;
                b[s] = src[s][inside ? xx : 0];
                b[s] = inside ? b[s] : 0.f;
            }
#pragma unroll
            for (int s = 0; s < STEPS; s++) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s], b[s], acc, 0, 0, 0);
            if (x0 + col >= D.X) continue;
            const long long at = vox(D, x0 + col, y, z) * CI + 4 * kg;
            *reinterpret_cast<float4 *>(gskip + at) = float4{acc[0], acc[1], acc[2], acc[3]};
            const uint2 m = *reinterpret_cast<const uint2 *>(act + at);
            float4 k;
            k.x = positive(m.x & 0xFFFFu) ? acc[0] : 0.f;
            k.y = positive(m.x >> 16) ? acc[1] : 0.f;
            k.z = positive(m.y & 0xFFFFu) ? acc[2] : 0.f;
            k.w = positive(m.y >> 16) ? acc[3] : 0.f;
            *reinterpret_cast<uint2 *>(gmask + at) = uint2{pack2(k.x, k.y), pack2(k.z, k.w)};
            sum.x += k.x;
            sum.y += k.y;
            sum.z += k.z;
            sum.w += k.w;
        }
    }
    __shared__ float s[4][CI];
    float v[4] = {sum.x, sum.y, sum.z, sum.w};
#pragma unroll
    for (int e = 0; e < 4; e++) {
        for (int off = 8; off > 0; off >>= 1) v[e] += __shfl_down(v[e], off, 16);
        if (col == 0) s[wave][4 * kg + e] = v[e];
    }
    __syncthreads();
    if (static_cast<int>(threadIdx.x) < CI)
        part[static_cast<size_t>(blockIdx.x) * CI + threadIdx.x] =
            (s[0][threadIdx.x] + s[1][threadIdx.x]) + (s[2][threadIdx.x] + s[3][threadIdx.x]);
}

// dL/dy of the mean squared error over n voxels; per workgroup the sum of
// (d^2) and of dL/dy (the last layer's bias gradient)
__global__ void __launch_bounds__(256) k_mse(long long n, const float *__restrict__ y,
                                             const float *__restrict__ target, float *__restrict__ gy,
                                             float *__restrict__ part) {
    float s = 0.f, b = 0.f;
    for (long long q = blockIdx.x * 256LL + threadIdx.x; q < n; q += 256LL * gridDim.x) {
        const float d = y[q] - target[q], g = 2.f * d / static_cast<float>(n);
        gy[q] = g;
        s += d * d;
        b += g;
    }
    group_sums(float4{s, b, 0.f, 0.f}, 1, part + 4 * static_cast<size_t>(blockIdx.x));
}

// out[job][c] = scale * sum over the job's rows of part[row * stride + c], a
// block of 64 columns per workgroup, its four wavefronts a quarter of the
// rows each, added in a fixed order
__global__ void __launch_bounds__(256) k_sum_rows(SumJobs J) {
    int q = 0, first = 0;
    for (; q < J.count - 1; q++) {
        const int blocks = (J.job[q].n + 63) / 64;
        if (static_cast<int>(blockIdx.x) < first + blocks) break;
        first += blocks;
    }
    const SumJob &job = J.job[q];
    const int c = (static_cast<int>(blockIdx.x) - first) * 64 + (threadIdx.x & 63), wave = threadIdx.x >> 6;
    __shared__ float s[4][64];
    float v = 0.f;
    if (c < job.n) {
        const int per = (job.rows + 3) / 4, r0 = wave * per, r1 = min(job.rows, r0 + per);
#pragma unroll 8
        for (int r = r0; r < r1; r++) v += job.part[static_cast<size_t>(r) * job.stride + c];
    }
    s[wave][threadIdx.x & 63] = v;
    __syncthreads();
    if (wave == 0 && c < job.n) {
        const int l = threadIdx.x;
        job.out[c] = job.scale * ((s[0][l] + s[1][l]) + (s[2][l] + s[3][l]));
    }
}

// Adam on all FP32 master parameters
__global__ void k_adam(int n, float *__restrict__ w, const float *__restrict__ g, float *__restrict__ m,
                       float *__restrict__ v, float lr, float b1, float b2, float eps, float c1, float c2) {
    const int q = blockIdx.x * 256 + threadIdx.x;
    if (q >= n) return;
    const float gq = g[q];
    const float mq = b1 * m[q] + (1.f - b1) * gq;
    const float vq = b2 * v[q] + (1.f - b2) * gq * gq;
    m[q] = mq;
    v[q] = vq;
    w[q] = w[q] - lr * (mq / c1) / (sqrtf(vq / c2) + eps);
}

// The BF16 copies of every layer's weights in one launch (blockIdx.y: layer).
// Plain layers: [27][ci][co] (data gradient) and [27][co][ci] (forward).
// Upsampling layers, whose weights on the coarse input are sums: with the
// fine taps t that meet on coarse tap t8 for output parity par (bits x, y, z
// from the lowest) added in FP32 in tap order, `fwd` is [par][t8][co][ci]
// (k_conv_fwd), rounded once, and `bwd` the sum of the BF16 weights as
// [3 terms][64 fine offsets][ci][co] (k_conv_up_dgrad): coarse tap o at parity
// p is the fine offset j = 3 - p - 2 o per axis, fine voxel 2 c - 1 + j.
__global__ void k_weights_bf16(WeightJobs J) {
    const WeightJob &l = J.job[blockIdx.y];
    const int ci = l.ci, co = l.co, n = (l.up ? 64 : 27) * ci * co;
    for (int q = blockIdx.x * 256 + threadIdx.x; q < n; q += 256 * gridDim.x) {
        if (!l.up) {
            const int t = q / (ci * co), r = q % (ci * co), i = r / co, o = r % co;
            const uint16_t b = f2bf(l.w[q]);
            l.bwd[q] = b;
            l.fwd[(t * co + o) * ci + i] = b;
            continue;
        }
        const int i = q % ci, o = (q / ci) % co, t8 = (q / (ci * co)) % 8, par = q / (8 * ci * co);
        const int p[3] = {par & 1, (par >> 1) & 1, par >> 2}, oo[3] = {t8 & 1, (t8 >> 1) & 1, t8 >> 2};
        float acc = 0.f, accb = 0.f;
        for (int t = 0; t < 27; t++) {
            int d[3];
            tap_offset(t, d[0], d[1], d[2]);
            bool hit = true;
            for (int a = 0; a < 3; a++) {
                const int c = (p[a] + d[a] + 2) / 2 - 1;  // floor((p + d) / 2)
                hit = hit && c == p[a] - 1 + oo[a];
            }
            if (hit) {
                const float w = l.w[(t * ci + i) * co + o];
                acc += w;
                accb += bf2f(f2bf(w));
            }
        }
        l.fwd[q] = f2bf(acc);
        const int jx = 3 - p[0] - 2 * oo[0], jy = 3 - p[1] - 2 * oo[1], jz = 3 - p[2] - 2 * oo[2];
        const int at = ((jx + 4 * jy + 16 * jz) * ci + i) * co + o;
        for (int h = 0; h < 3; h++) {
            const uint16_t term = f2bf(accb);
            l.bwd[64 * h * ci * co + at] = term;
            accb -= bf2f(term);  // exact
        }
    }
}

inline unsigned blocks_for(long long n) {
    const long long b = (n + 255) / 256;
    return static_cast<unsigned>(b > 8192 ? 8192 : (b < 1 ? 1 : b));
}

}  // namespace

// ---------------------------------------------------------------- launchers
#define ARTSS_CONV_CASES(X) X(16, 32) X(32, 64) X(64, 64) X(64, 32) X(32, 16)
// voxels per wavefront row of k_conv_fwd: 16 x NV, eight matrix tiles per K step
constexpr int row_tiles(int co) { return co == 16 ? 8 : (co == 32 ? 4 : 2); }

// Planes per wavefront of the marching kernels, for `columns` wavefronts per
// plane of `z`: four wavefronts per SIMD if the volume has them, within 4
// planes (half the planes read are then halo) and 16
int march_planes(long long columns, int z) {
    const long long p = z * columns / 4096;
    return static_cast<int>(std::min(16LL, std::max(4LL, p)));
}
template <bool GRAD>
void launch_conv16(hipStream_t s, Dims D, const uint16_t *in, const uint16_t *Wt, const float *bias, uint16_t *out,
                   uint16_t *pre, const uint16_t *skip, bool relu, float *gin) {
    const int gx = (D.X + 15) / 16, gy = (D.Y + 4 * kRows16 - 1) / (4 * kRows16);
    const int planes = march_planes(4LL * gx * gy, D.Z);
    k_conv16<GRAD><<<dim3(gx, gy, (D.Z + planes - 1) / planes), 256, 0, s>>>(D, in, Wt, bias, out, pre, skip, relu ? 1 : 0,
                                                                            gin, planes);
}

void conv_fwd(hipStream_t s, int cin, int cout, bool up, Dims D, const uint16_t *in, const uint16_t *Wt,
              const float *bias, uint16_t *out, uint16_t *pre, const uint16_t *skip, bool relu) {
    if (cin == 16 && cout == 16 && !up) {
        launch_conv16<false>(s, D, in, Wt, bias, out, pre, skip, relu, nullptr);
        return;
    }
    if (cin == 32 && cout == 16 && up) {
        const int cx = D.X >> 1, cy = D.Y >> 1, cz = D.Z >> 1;
        const int gx = (cx + 15) / 16, gy = (cy + 7) / 8, planes = march_planes(4LL * gx * gy, cz);
        const int gz = (cz + planes - 1) / planes;
        // two workgroups of its 64 KiB fit a CU: it needs about that many to
        // beat k_conv_fwd (256x128x128, 1024 workgroups: 170 against 199 us;
        // 128x64x64, 128 workgroups: 59 against 32 us)
        if (gx * gy * gz >= 512) {
            k_conv_up16<<<dim3(gx, gy, gz), 256, 0, s>>>(D, in, Wt, bias, out, pre, skip, relu ? 1 : 0, planes);
            return;
        }
    }
#define CASE(CI, CO)                                                                                             \
    if (cin == CI && cout == CO) {                                                                              \
        constexpr int NV = row_tiles(CO);                                                                       \
        const dim3 g((D.X + 16 * NV - 1) / (16 * NV), (D.Y + 3) / 4, D.Z);                                     \
        if (!up) {                                                                                              \
            k_conv_fwd<CI, CO, false, NV>                                                                       \
                <<<g, 256, 0, s>>>(D, in, Wt, bias, out, pre, skip, relu ? 1 : 0, nullptr);                     \
            return;                                                                                             \
        }                                                                                                       \
        if constexpr (CI >= 32) {                                                                               \
            k_conv_fwd<CI, CO, true, NV>                                                                        \
                <<<g, 256, 0, s>>>(D, in, Wt, bias, out, pre, skip, relu ? 1 : 0, nullptr);                     \
            return;                                                                                             \
        }                                                                                                       \
        throw std::invalid_argument("conv_fwd: an upsampled input needs at least 32 channels");               \
    }
    ARTSS_CONV_CASES(CASE)
#undef CASE
    throw std::invalid_argument("conv_fwd: unsupported channel pair");
}

void conv_dgrad(hipStream_t s, int cin, int cout, Dims D, const uint16_t *g, const uint16_t *W, const uint16_t *act,
                float *gin) {
    if (cin == 16 && cout == 16) {
        launch_conv16<true>(s, D, g, W, nullptr, nullptr, nullptr, act, false, gin);
        return;
    }
#define CASE(CI, CO)                                                                                             \
    if (cin == CI && cout == CO) {                                                                              \
        constexpr int NV = row_tiles(CI);                                                                       \
        const dim3 grid((D.X + 16 * NV - 1) / (16 * NV), (D.Y + 3) / 4, D.Z);                                  \
        k_conv_fwd<CO, CI, false, NV, true>                                                                     \
            <<<grid, 256, 0, s>>>(D, g, W, nullptr, nullptr, nullptr, act, 0, gin);                             \
        return;                                                                                                 \
    }
    CASE(16, 32) CASE(32, 64) CASE(64, 64)
#undef CASE
    throw std::invalid_argument("conv_dgrad: unsupported channel pair");
}

int up_dgrad_rows(int cin, int cout, Dims Dc) {
    const int nv = cout == 64 ? 1 : (cin == 64 ? 2 : 4);
    const long long tiles = static_cast<long long>((Dc.X + 16 * nv - 1) / (16 * nv)) * Dc.Y * Dc.Z;
    return static_cast<int>(tiles < 1024 ? tiles : 1024);
}
void conv_up_dgrad(hipStream_t s, int cin, int cout, Dims Dc, const uint16_t *g, const uint16_t *Wd,
                   const uint16_t *act, float *gskip, uint16_t *gmask, float *part) {
    const unsigned rows = static_cast<unsigned>(up_dgrad_rows(cin, cout, Dc));
    if (cin == 32 && cout == 16) k_conv_up_dgrad<16, 32, 4, 4, 2><<<rows, 256, 0, s>>>(Dc, g, Wd, act, gskip, gmask, part);
    else if (cin == 64 && cout == 32)
        k_conv_up_dgrad<32, 64, 2, 4, 4><<<rows, 256, 0, s>>>(Dc, g, Wd, act, gskip, gmask, part);
    else if (cin == 64 && cout == 64)
        k_conv_up_dgrad<64, 64, 1, 8, 1><<<dim3(rows, 4), 512, 0, s>>>(Dc, g, Wd, act, gskip, gmask, part);
    else throw std::invalid_argument("conv_up_dgrad: unsupported channel pair");
}

// Partial rows of a weight gradient: enough workgroups (x 3 z offsets) to
// fill the chip, few enough that the rows written and added again stay a
// small part of the pass (27 ci co floats each).
int wgrad_rows(int cin, int cout, Dims D) {
    const int most = cin * cout <= 512 ? 256 : (cin * cout <= 2048 ? 96 : 32);
    const int blocks = grad_blocks(D).blocks;
    return blocks < most ? blocks : most;
}
void conv_wgrad(hipStream_t s, int cin, int cout, bool up, Dims D, const uint16_t *in, const uint16_t *g,
                float *part) {
    const GradBlocks B = grad_blocks(D);
    const dim3 grid(static_cast<unsigned>(wgrad_rows(cin, cout, D)), 3);
    const size_t fmax = static_cast<size_t>((B.rows * B.xb + 31) & ~31);
    const size_t pos = up ? static_cast<size_t>(B.rows / 2 + 2) * ((B.xb + 1) / 2 + 2)
                          : static_cast<size_t>(B.rows + 2) * (B.xb + 2);
#define CASE(CI, CO, UP)                                                                                       \
    if (cin == CI && cout == CO && up == UP) {                                                                \
        const size_t bytes = 2 * (fmax * lds_voxel<CO>() + pos * lds_voxel<CI>());                            \
        /* at most (2 + 2) x (128 + 2) halo voxels and 256 others: 121 KB at 64 channels */                   \
        if (bytes > 64 * 1024 &&                                                                              \
            hipFuncSetAttribute(reinterpret_cast<const void *>(&k_conv_wgrad<CI, CO, UP>),                    \
                                hipFuncAttributeMaxDynamicSharedMemorySize,                                   \
                                static_cast<int>(bytes)) != hipSuccess)                                       \
            throw std::runtime_error("conv_wgrad: the block does not fit in this device's LDS");              \
        k_conv_wgrad<CI, CO, UP><<<grid, 192, bytes, s>>>(D, B, in, g, part);                                 \
        return;                                                                                               \
    }
    CASE(16, 16, false) CASE(16, 32, false) CASE(32, 64, false) CASE(64, 64, false)
    CASE(64, 64, true) CASE(64, 32, true) CASE(32, 16, true)
#undef CASE
    throw std::invalid_argument("conv_wgrad: unsupported channel pair");
}

void conv_in(hipStream_t s, Dims D, const float *x, const float *W, const float *bias, uint16_t *out) {
    const int gx = (D.X + 15) / 16, gy = (D.Y + 4 * kRows16 - 1) / (4 * kRows16);
    const int planes = march_planes(4LL * gx * gy, D.Z);
    k_conv_in<<<dim3(gx, gy, (D.Z + planes - 1) / planes), 256, 0, s>>>(D, x, W, bias, out, planes);
}
void conv_out(hipStream_t s, Dims D, const uint16_t *in, const float *W, const float *bias, float *y) {
    k_conv_out<16, 8><<<dim3((D.X + 63) / 64, (D.Y + 3) / 4, (D.Z + 7) / 8), dim3(64, 4, 1), 0, s>>>(D, in, W, bias, y);
}
// one workgroup per four x rows, at most two per CU
int end_wgrad_rows(Dims D) {
    const long long lines = static_cast<long long>(D.Y) * D.Z;
    return static_cast<int>(lines < 4 * 512 ? (lines + 3) / 4 : 512);
}
void conv_in_wgrad(hipStream_t s, Dims D, const float *x, const float *g, float *part) {
    k_conv_in_wgrad<<<static_cast<unsigned>(end_wgrad_rows(D)), 256, 0, s>>>(D, x, g, part);
}
void conv_out_wgrad(hipStream_t s, Dims D, const uint16_t *in, const float *gy, float *part) {
    k_conv_out_wgrad<<<static_cast<unsigned>(end_wgrad_rows(D)), 256, 0, s>>>(D, in, gy, part);
}
int end_dgrad_rows(Dims D) {
    const long long lines = static_cast<long long>(D.Y) * D.Z;
    return static_cast<int>(lines < 4 * 1024 ? (lines + 3) / 4 : 1024);
}
int elementwise_rows(long long voxels, int groups) {
    const long long b = (voxels * groups + 1023) / 1024;  // four items per thread
    return static_cast<int>(b < 1 ? 1 : (b > 512 ? 512 : b));
}
void conv_out_dgrad(hipStream_t s, Dims D, const float *W, const float *gy, const uint16_t *act, float *gskip,
                    uint16_t *gmask, float *part) {
    k_conv_out_dgrad<16><<<static_cast<unsigned>(end_dgrad_rows(D)), 256, 0, s>>>(D, W, gy, act, gskip, gmask, part);
}
void enc_grad(hipStream_t s, int c, Dims D, const float *gskip, const float *gc, const uint16_t *act, uint16_t *gmask,
              float *part) {
    const unsigned b = static_cast<unsigned>(elementwise_rows(static_cast<long long>(D.X) * D.Y * D.Z, c / 4));
    if (c == 16) k_enc_grad<16><<<b, 256, 0, s>>>(D, gskip, gc, act, gmask, part);
    else if (c == 32) k_enc_grad<32><<<b, 256, 0, s>>>(D, gskip, gc, act, gmask, part);
    else if (c == 64) k_enc_grad<64><<<b, 256, 0, s>>>(D, gskip, gc, act, gmask, part);
    else throw std::invalid_argument("enc_grad: unsupported channels");
}
void down(hipStream_t s, int c, Dims Dc, const uint16_t *in, uint16_t *out) {
    const long long n = static_cast<long long>(Dc.X) * Dc.Y * Dc.Z * c;
    if (c == 16) k_down<16><<<blocks_for(n), 256, 0, s>>>(Dc, in, out);
    else if (c == 32) k_down<32><<<blocks_for(n), 256, 0, s>>>(Dc, in, out);
    else if (c == 64) k_down<64><<<blocks_for(n), 256, 0, s>>>(Dc, in, out);
    else throw std::invalid_argument("down: unsupported channels");
}
void mse(hipStream_t s, long long n, const float *y, const float *target, float *gy, float *part) {
    k_mse<<<static_cast<unsigned>(elementwise_rows(n, 1)), 256, 0, s>>>(n, y, target, gy, part);
}
void sum_rows(hipStream_t s, const SumJobs &jobs) {
    unsigned blocks = 0;
    for (int q = 0; q < jobs.count; q++) blocks += static_cast<unsigned>((jobs.job[q].n + 63) / 64);
    if (blocks) k_sum_rows<<<blocks, 256, 0, s>>>(jobs);
}
void adam(hipStream_t s, int n, float *w, const float *g, float *m, float *v, float lr, float b1, float b2, float eps,
          float c1, float c2) {
    k_adam<<<static_cast<unsigned>((n + 255) / 256), 256, 0, s>>>(n, w, g, m, v, lr, b1, b2, eps, c1, c2);
}
void weights_bf16(hipStream_t s, const WeightJobs &jobs) {
    if (jobs.count) k_weights_bf16<<<dim3(256, static_cast<unsigned>(jobs.count)), 256, 0, s>>>(jobs);
}

}  // namespace nn
}  // namespace artss
