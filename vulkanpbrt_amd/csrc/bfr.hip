// BFR (blockwise feature regression fitted by Adam) and the three-size blender
// on gfx950.
//
// bfr.comp fits, per b x b block, a 7-feature linear model of the accumulated
// demodulated illumination,
//   features [1, sx, sy, 2 z - 1, n.x, n.y, n.z]   (sx, sy in [-0.5, 0.5] over the
//   block, z = per-block normalised depth), alpha: 7 x rgb
// by 40 steps of Adam on the block-summed residual gradient (plain residual, or its
// sign once a pixel has >= 10 samples; the optimiser constants blend between the
// two regimes by the fraction of such pixels), then reconstructs, blends with the
// reprojected previous output and remodulates (bfr.comp:202-308).
//
// The reference runs one b x b workgroup per block (up to 1024 threads) with two
// barriers per Adam step.  Here a 16- or 8-pixel block is one wave and a 32-pixel block
// four: a step forms the 21 gradient sums of each 64-pixel group with lane swaps (two
// sums share a register at xor 32, four at xor 16), lane j of the wave then runs
// Adam for component j alone and the 21 new weights go to scalar registers.
//
// Project rules where bfr.comp depends on the hardware:
//   * the stop test `gradient_rest >= GRADIENT_THRESH (0)` is reduced over all 7
//     alpha components (bfr.comp takes a subgroup-dependent subset); it only ends
//     the loop early when the gradient is NaN.
//   * sums run in a fixed wave / lane tree order (the reference's subgroup order is
//     vendor-specific); results agree with the oracle to fp32 rounding.
#include <hip/hip_runtime.h>

#include "capi_common.hpp"
#include "image_ops.hpp"
#include "wave_sums.hpp"

namespace pbrt {

namespace {

constexpr int kBfrFeatures = 7;
constexpr int kBfrSums = 3 * kBfrFeatures;  // gradient components per step
constexpr int kBfrIterations = 40;          // GRADIENT_ITERATION_AMT

// Adam constants of bfr.comp:77-88
constexpr float kAlpha = 0.863f, kK = 0.116f, kBeta1 = 0.3f, kBeta2 = 0.7314f, kEps = 1e-8f;
constexpr float kAlphaL = 1.1f, kBeta1L = 0.45f, kBeta2L = 0.75f;
constexpr float kSppThreshold = 10.0f;

// pixelOffsets of bfr.comp:92 (integer, added to the invocation position)
const int kBfrOffsetsHost[16][2] = {{-7, -11}, {-14, -8}, {-5, -12}, {-15, -1}, {-5, -9},  {-1, -4},
                                    {-14, -7}, {0, -13},  {-5, -1},  {-1, 0},   {-15, -2}, {-14, -10},
                                    {-1, -1},  {-6, -3},  {0, -8},   {-10, -4}};

struct BfrGeom {
    int width, height, bs, blocks_x, blocks_y, offx, offy;
    uint32_t frame;
};

__device__ __forceinline__ float wave_min(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fminf(v, __shfl_xor(v, off));
    return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off));
    return v;
}

__device__ __forceinline__ float sign_of(float x) { return x > 0.0f ? 1.0f : (x < 0.0f ? -1.0f : 0.0f); }

}  // namespace

// The step loop is VALU-bound: per 64 pixels 21 multiply-adds of prediction, 21 of
// gradient and the signs, and then the 21 sums.  What it spends beside them is kept off
// the vector unit's redundant lanes:
//   * the sums: v_permlane32_swap / v_permlane16_swap exchange half a register with
//     another sum's, so xor 32 and 16 cost one swap and one add per two sums (plain
//     butterflies through the LDS pipe: two operations per sum and step, 126 per wave
//     and iteration in all), and xor 8 and 4 are row rotations (DPP);
//   * Adam once per component in lane j instead of all 21 components in every lane (a
//     correctly rounded square root and division each), its learning-rate factors from
//     a table made once per block, lane t holding step t;
//   * the new weights by v_readlane into scalar registers, which the multiply-adds read.
// A sum is the same binary tree over the same pixels as a butterfly from xor 32 to xor 1
// followed by the 64-pixel groups in order, so the steps' signs do not change with the
// mapping.  One wave per 16-pixel block (four groups a lane) needs no barrier and runs
// the sums' rows, Adam and the broadcast once instead of four times; a 32-pixel block's
// 16 pixels per lane would leave two waves per SIMD, so it takes four waves and one
// barrier a step.  At 1920x1080: 16-pixel blocks 2402 -> 357 us, 8-pixel 2335 -> 444 us,
// 32-pixel 835 -> 246 us.
constexpr int kSumSlots = 24;  // 21 gradient components, padded

// kB: block edge; kW waves per block; a lane owns kP pixels of each of kV groups of 64:
// pixel r = (wave * kV + group) * 64 + lane + p * 64 kW kV at local (r / kB, r % kB)
// (bfr.comp's ID order).
template <int kB, int kW, int kV, int kP>
__global__ void __launch_bounds__(64 * kW) k_bfr(BfrGeom g, pbrt_bfr_images im) {
    constexpr int kPix = kV * kP;
    static_assert(64 * kW * kPix == kB * kB, "the lanes' pixels are the block's");
    static_assert(kW == 1 || kV == 1, "a sum has four parts at most");
    constexpr int kParts = kW * kV;  // 64-lane partial sums per component: 1 or 4
    static_assert(kParts == 1 || kParts == 4, "parts are read as one or four floats");
    __shared__ __attribute__((aligned(16))) float part[kW > 1 ? 2 : 1][kSumSlots * kParts];
    __shared__ float red[3][kW];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

    vec3 color[kPix];
    float feat[kPix][kBfrFeatures];
    bool l1px[kPix];
    int img_x[kPix], img_y[kPix];
    bool inside[kPix];
    float depth[kPix];
    float dmin = 3.4e38f, dmax = -3.4e38f;
    int l1_count = 0;
#pragma unroll
    for (int p = 0; p < kPix; ++p) {
        const int r = (wave * kV + p / kP) * 64 + lane + (p % kP) * 64 * kParts;
        const int lx = r / kB, ly = r % kB;
        const int ax = blockIdx.x * kB + lx + g.offx, ay = blockIdx.y * kB + ly + g.offy;
        img_x[p] = mirror_coord(ax, g.width);
        img_y[p] = mirror_coord(ay, g.height);
        inside[p] = ax == img_x[p] && ay == img_y[p];
        const size_t pix = (size_t)img_y[p] * g.width + img_x[p];
        color[p] = xyz(load_half4(im.noisy, pix));
        depth[p] = im.depth[pix];
        const float2 n = reinterpret_cast<const float2*>(im.normal)[pix];
        const vec3 nn = decode_normal(n.x, n.y);
        const float spp = unorm8_to_float(im.spp[pix]) * 256.0f;
        l1px[p] = spp >= kSppThreshold;
        l1_count += __popcll(__ballot(l1px[p]));
        dmin = fminf(dmin, depth[p]);
        dmax = fmaxf(dmax, depth[p]);
        feat[p][0] = 1.0f;
        feat[p][1] = (float)lx / (float)(kB - 1) - 0.5f;
        feat[p][2] = (float)ly / (float)(kB - 1) - 0.5f;
        feat[p][4] = nn.x;
        feat[p][5] = nn.y;
        feat[p][6] = nn.z;
    }
    // block min / max depth and the count of pixels in the L1 regime
    dmin = wave_min(dmin);
    dmax = wave_max(dmax);
    float l1f = (float)l1_count;
    if (kW > 1) {
        if (lane == 0) {
            red[0][wave] = dmin;
            red[1][wave] = dmax;
            red[2][wave] = l1f;
        }
        __syncthreads();
        dmin = red[0][0];
        dmax = red[1][0];
        l1f = red[2][0];
#pragma unroll
        for (int w = 1; w < kW; ++w) {
            dmin = fminf(dmin, red[0][w]);
            dmax = fmaxf(dmax, red[1][w]);
            l1f += red[2][w];
        }
    }
#pragma unroll
    for (int p = 0; p < kPix; ++p) {
        float z = depth[p] - dmin;
        z /= dmax - dmin + kEps;
        feat[p][3] = z * 2.0f - 1.0f;
    }
    const float l1_ratio = l1f * 1.0f / (float)(kB * kB);
    const float a_mix = l1_ratio * kAlphaL + (1.0f - l1_ratio) * kAlpha;
    const float b1_mix = l1_ratio * kBeta1L + (1.0f - l1_ratio) * kBeta1;
    const float b2_mix = l1_ratio * kBeta2L + (1.0f - l1_ratio) * kBeta2;
    // exponential learning-rate decay and bias correction (bfr.comp:124-131) of step
    // t = lane + 1
    const float t_lane = (float)(lane + 1);
    const float step_lane =
        a_mix * expf(-kK * t_lane) * sqrtf(1.0f - powf(kBeta2, t_lane)) / (1.0f - powf(kBeta1, t_lane));

    // lane j: component j of alpha and of Adam's moments; aw: alpha on every lane
    float alpha_lane = 0.0f, m = 0.0f, v = 0.0f;
    float aw[kBfrSums];
#pragma unroll
    for (int j = 0; j < kBfrSums; ++j) aw[j] = 0.0f;

    const int row = lane >> 4, bank = (lane >> 2) & 3, quad = lane & 3;
    for (int it = 0; it < kBfrIterations; ++it) {
        float grad[kV][kBfrSums];
#pragma unroll
        for (int w = 0; w < kV; ++w)
#pragma unroll
            for (int j = 0; j < kBfrSums; ++j) grad[w][j] = 0.0f;
#pragma unroll
        for (int p = 0; p < kPix; ++p) {
            vec3 pred = make_vec3(0.0f);
#pragma unroll
            for (int j = 0; j < kBfrFeatures; ++j)
                pred += make_vec3(aw[3 * j], aw[3 * j + 1], aw[3 * j + 2]) * feat[p][j];
            vec3 d = color[p] - pred;
            if (l1px[p]) d = make_vec3(sign_of(d.x), sign_of(d.y), sign_of(d.z));
            float* gw = grad[p / kP];
#pragma unroll
            for (int j = 0; j < kBfrFeatures; ++j) {
                gw[3 * j] += feat[p][j] * d.x;
                gw[3 * j + 1] += feat[p][j] * d.y;
                gw[3 * j + 2] += feat[p][j] * d.z;
            }
        }
        float* slot = part[kW > 1 ? (it & 1) : 0];
        if constexpr (kV == 4) {
            // row r: group r's part of a component; four components by lane quartet (bank),
            // four such registers by lane within the quartet
            float q[kSumSlots / 4];
#pragma unroll
            for (int f = 0; f < kSumSlots / 4; ++f) {
                float s[4];
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    const int j = 4 * f + b;
                    s[b] = 0.0f;
                    if (j < kBfrSums) s[b] = row_steps84(rows_of(grad[0][j], grad[1][j], grad[2][j], grad[3][j]));
                }
                q[f] = quad_steps21(by_bank(bank, s[0], s[1], s[2], s[3]));
            }
            slot[(4 * quad + bank) * 4 + row] = by_bank(quad, q[0], q[1], q[2], q[3]);
            if (quad < 2) slot[(16 + 4 * quad + bank) * 4 + row] = quad ? q[5] : q[4];
        } else {
            // row r: component 4 k + r of register k, the lane's by its quartet
            float q[kSumSlots / 4];
#pragma unroll
            for (int k = 0; k < kSumSlots / 4; ++k) {
                float s[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) s[r] = 4 * k + r < kBfrSums ? grad[0][4 * k + r] : 0.0f;
                q[k] = row_steps84(rows_of(s[0], s[1], s[2], s[3]));
            }
            const float a = quad_steps21(by_bank(bank, q[0], q[1], q[2], q[3]));
            const float b = quad_steps21((bank & 1) ? q[5] : q[4]);
            if (quad == 0) {
                slot[(4 * bank + row) * kParts + wave] = a;
                if (bank < 2) slot[(16 + 4 * bank + row) * kParts + wave] = b;
            }
        }
        if (kW > 1)
            __syncthreads();
        else
            wave_lds_sync();
        float gj = 0.0f;
        if (lane < kBfrSums) {
            if constexpr (kParts == 4) {
                const float4 s = *reinterpret_cast<const float4*>(slot + 4 * lane);
                gj = s.x + s.y + s.z + s.w;
            } else {
                gj = slot[lane];
            }
        }
        if (kW == 1) wave_lds_sync();  // one slot: read before the next step's sums are written
        const float step = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(step_lane), it));
        m = b1_mix * m + (1.0f - kBeta1) * gj;
        v = b2_mix * v + (1.0f - kBeta2) * (gj * gj);
        alpha_lane += step * (m / (sqrtf(v) + kEps));
#pragma unroll
        for (int j = 0; j < kBfrSums; ++j)
            aw[j] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(alpha_lane), j));
        if (__any(gj != gj)) break;  // NaN gradient (GRADIENT_THRESH = 0)
    }

    if (im.weights && tid < kBfrSums)
        im.weights[((size_t)blockIdx.y * g.blocks_x + blockIdx.x) * kBfrSums + tid] = alpha_lane;

    const size_t plane = (size_t)g.width * g.height;
#pragma unroll
    for (int p = 0; p < kPix; ++p) {
        if (!inside[p]) continue;
        const size_t pix = (size_t)img_y[p] * g.width + img_x[p];
        vec3 den = make_vec3(0.0f);
#pragma unroll
        for (int j = 0; j < kBfrFeatures; ++j)
            den += make_vec3(aw[3 * j], aw[3 * j + 1], aw[3 * j + 2]) * feat[p][j];
        den = vclamp(den, 0.0f, 10.0f);
        const ushort2 mv = reinterpret_cast<const ushort2*>(im.motion)[pix];
        const float mux = h2f(mv.x), muy = h2f(mv.y);
        vec3 prev = make_vec3(0.0f);
        float blend = 1.0f;
        if (g.frame > 0 && mux >= 0.0f) {
            const uint16_t* layer = im.denoised + 4 * plane * (g.frame & 1u);
            const int w = g.width;
            prev = xyz(sample_bilinear([&](int sx, int sy) { return load_half4(layer, (size_t)sy * w + sx); },
                                       g.width, g.height, mux, muy));
            const float spp = unorm8_to_float(im.spp[pix]) * 256.0f;
            blend = fmaxf(1.0f / spp, 0.1f);
        }
        den = blend * den + (1.0f - blend) * prev;
        store_half4(im.denoised + 4 * plane * ((g.frame & 1u) ^ 1u), pix, make_vec4(den, 1.0f));
        const vec3 alb = xyz(load_rgba8(im.albedo, pix)) + make_vec3(1e-6f);
        vec3 tm = alb * den;
        tm = make_vec3(fmaxf(tm.x, 0.0f), fmaxf(tm.y, 0.0f), fmaxf(tm.z, 0.0f));
        tm = vclamp(vpow(tm, 0.454545f), 0.0f, 1.0f);
        store_bgra8(im.final_image, pix, make_vec4(tm, 1.0f));
    }
}

// mix3 of bfrBlender.comp:19-27
__device__ __forceinline__ float mix3(float a, float b, float c, float t, float mid, float max_dev) {
    t /= max_dev;
    t = fminf(t, 1.0f);  // a NaN deviation selects t = 1 (IEEE minNum)
    const float fa = fmaxf(1.0f - (t / mid), 0.0f);
    const float fb = (t < mid) ? t / mid : 1.0f - (t - mid) / (1.0f - mid);
    const float fc = 1.0f - fa - fb;
    return fa * a + fb * b + fc * c;
}

__device__ __forceinline__ float glsl_mix(float x, float y, float a) { return x * (1.0f - a) + y * a; }

__global__ void __launch_bounds__(256) k_bfr_blend(int w, int h, int radius, pbrt_bfr_blend_images im) {
    const int x = blockIdx.x * 16 + (threadIdx.x & 15), y = blockIdx.y * 16 + (threadIdx.x >> 4);
    if (x >= w || y >= h) return;
    float sq = 0.0f, av = 0.0f;
    int count = 0;
    for (int dy = -radius; dy <= radius; ++dy)
        for (int dx = -radius; dx <= radius; ++dx) {
            const int sx = x + dx, sy = y + dy;
            vec3 a = make_vec3(0.0f);
            if (sx >= 0 && sy >= 0 && sx < w && sy < h) a = xyz(load_half4(im.average, (size_t)sy * w + sx));
            const float cur = dot(a, make_vec3(1.0f / 3.0f));
            ++count;
            sq = glsl_mix(sq, cur * cur, 1.0f / (float)count);
            av = glsl_mix(av, cur, 1.0f / (float)count);
        }
    const size_t pix = (size_t)y * w + x;
    const vec3 ave = xyz(load_half4(im.average, pix));
    const vec3 ave2 = xyz(load_half4(im.average_squared, pix));
    av = glsl_mix(av, dot(ave, make_vec3(1.0f / 3.0f)), 0.5f);
    sq = glsl_mix(sq, dot(ave2, make_vec3(1.0f / 3.0f)), 0.5f);
    // bfrBlender.comp loads denoised0 (8x8) into den2 and denoised2 (32x32) into den0
    const vec3 den2 = xyz(load_bgra8(im.denoised8, pix));
    const vec3 den1 = xyz(load_bgra8(im.denoised16, pix));
    const vec3 den0 = xyz(load_bgra8(im.denoised32, pix));
    const float sd = sqrtf(sq - av * av);
    const vec3 c = make_vec3(mix3(den0.x, den1.x, den2.x, sd, 0.5f, 1.0f), mix3(den0.y, den1.y, den2.y, sd, 0.5f, 1.0f),
                             mix3(den0.z, den1.z, den2.z, sd, 0.5f, 1.0f));
    store_bgra8(im.final_image, pix, make_vec4(c, 1.0f));
}

}  // namespace pbrt

using namespace pbrt;

extern "C" int32_t pbrt_bfr(const pbrt_bfr_params* p, const pbrt_bfr_images* im, void* stream) {
    return guard([&] {
        PBRT_REQUIRE(p && im, "pbrt_bfr: NULL argument");
        PBRT_REQUIRE(p->block_size == 8 || p->block_size == 16 || p->block_size == 32,
                     "pbrt_bfr: block_size must be 8, 16 or 32");
        PBRT_REQUIRE(p->width >= 2 * p->block_size && p->height >= 2 * p->block_size && p->width >= 16 &&
                         p->height >= 16,
                     "pbrt_bfr: image must be at least two blocks (and 16 pixels) wide and high (mirror addressing)");
        PBRT_REQUIRE(im->depth && im->normal && im->albedo && im->motion && im->spp && im->noisy && im->denoised &&
                         im->final_image,
                     "pbrt_bfr: NULL image");
        BfrGeom g{};
        g.width = (int)p->width;
        g.height = (int)p->height;
        g.bs = (int)p->block_size;
        g.blocks_x = g.width / g.bs + 2;
        g.blocks_y = g.height / g.bs + 2;
        g.offx = kBfrOffsetsHost[p->frame_number % 16][0];
        g.offy = kBfrOffsetsHost[p->frame_number % 16][1];
        g.frame = p->frame_number;
        const dim3 grid(g.blocks_x, g.blocks_y);
        hipStream_t st = (hipStream_t)stream;
        if (g.bs == 8)
            hipLaunchKernelGGL((k_bfr<8, 1, 1, 1>), grid, dim3(64), 0, st, g, *im);
        else if (g.bs == 16)
            hipLaunchKernelGGL((k_bfr<16, 1, 4, 1>), grid, dim3(64), 0, st, g, *im);
        else
            hipLaunchKernelGGL((k_bfr<32, 4, 1, 4>), grid, dim3(256), 0, st, g, *im);
        PBRT_HIP(hipGetLastError());
    });
}

extern "C" int32_t pbrt_bfr_blend(uint32_t width, uint32_t height, uint32_t filter_radius,
                                  const pbrt_bfr_blend_images* im, void* stream) {
    return guard([&] {
        PBRT_REQUIRE(im && im->average && im->average_squared && im->denoised8 && im->denoised16 &&
                         im->denoised32 && im->final_image,
                     "pbrt_bfr_blend: NULL image");
        PBRT_REQUIRE(filter_radius <= 16, "pbrt_bfr_blend: filter_radius above 16");
        if (width == 0 || height == 0) return;
        const dim3 grid((width + 15) / 16, (height + 15) / 16);
        hipLaunchKernelGGL(k_bfr_blend, grid, dim3(256), 0, (hipStream_t)stream, (int)width, (int)height,
                           (int)filter_radius, *im);
        PBRT_HIP(hipGetLastError());
    });
}
