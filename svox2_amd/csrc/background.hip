// The MSI background (multi-sphere image) composited behind the grid, its
// gradients, and its total variation.
//
// The background is nlayers concentric spheres around the grid's unit sphere,
// each an equirectangular image of [2 reso][reso] pixels holding (r, g, b,
// sigma); links map a pixel column to a row of background_data
// ([rows][nlayers] float4), -1 = empty.  A ray leaving the grid with log
// transmittance log_t (the grid's own, rendered with background brightness 0)
// samples the spheres at radii n_steps / (n_steps - i - 0.5), i = 0 ..
// n_steps - 1 (n_steps = nlayers / step_size + 2), from the inside out; each
// sample is trilinear in (longitude, latitude, layer), its step is the change
// of 1 / radius times the ray's world step, and it composites like the grid's
// samples (render_background_forward / _backward,
// render_lerp_kernel_cuvol.cu:386-607; kernels :775-860).  The transmittance
// left after the last layer sees the background brightness.
//
// One 32-lane group per ray, one lane per sample: a chunk of 32 samples is
// placed and read in parallel (8 float4 loads per sample: 4 pixel columns x 2
// layers, all four channels at once), its transmittance is an inclusive scan
// of the samples' optical depths, and the stop threshold cuts the chunk at the
// first sample whose transmittance falls below it.  The reference walks the
// samples one by one in a thread per ray; the sums here are the same terms
// added in scan order.  The backward then adds the samples in march order into
// registers, a lane per (grid point, channel), and writes a grid point out when
// the ray leaves it.
#include "common.hpp"

namespace svox2amd {
namespace {

constexpr int kBgBlock = 256;
constexpr int kBgGroup = 32;
constexpr float kShC0 = 0.28209479177387814f;
constexpr float kInvPi = 0.318309886183790671538f;

struct BgView {
    const int32_t* links;  // [2 reso][reso]
    const float4* data;    // [rows * nlayers]
    float* grad;           // [rows * nlayers * 4] (backward)
    uint8_t* mask;         // [rows * nlayers] (backward, may be NULL)
    int64_t rows;
    int reso, nlayers, n_steps;
    float offset[3], scaling[3], sph[3];  // sph = 2 / grid size
    float bg, stop;                       // background brightness, stop threshold
};

// The ray in the frame where the grid's sphere is the unit sphere
// (ray_find_bounds_bg, render_util.cuh:630-657), and its sphere
// intersection coefficients (ConcentricSpheresIntersector, :546-576).
struct BgRay {
    float o[3], d[3];
    float ws;     // world length per unit of (1 / radius) change
    float q2a, qb, f;
    float inner;  // first radius: max(distance of the line to the centre + 1e-3, 1)
};

__device__ __forceinline__ float bg_dot(const float* a, const float* b) {
    return a[0] * b[0] + a[1] * b[1] + a[2] * b[2];
}

__device__ __forceinline__ void bg_ray(const BgView& b, const float* wo, const float* wd,
                                       BgRay& r) {
    float o[3], d[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        o[i] = fmaf(wo[i], b.scaling[i], b.offset[i]);
        d[i] = wd[i] * b.scaling[i];
    }
    float ws = 1.0f / sqrtf(bg_dot(d, d));
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        d[i] *= ws;
        r.o[i] = fmaf(o[i] + 0.5f, b.sph[i], -1.f);
        r.d[i] = d[i] * b.sph[i];
    }
    const float inorm = 1.0f / sqrtf(bg_dot(r.d, r.d));
    r.ws = ws * inorm;
#pragma unroll
    for (int i = 0; i < 3; ++i) r.d[i] *= inorm;
    r.q2a = 2.f * bg_dot(r.d, r.d);
    r.qb = 2.f * bg_dot(r.o, r.d);
    r.f = r.qb * r.qb - 2.f * r.q2a * bg_dot(r.o, r.o);
    const float cx = r.o[1] * r.d[2] - r.o[2] * r.d[1];
    const float cy = r.o[2] * r.d[0] - r.o[0] * r.d[2];
    const float cz = r.o[0] * r.d[1] - r.o[1] * r.d[0];
    r.inner = fmaxf(sqrtf(cx * cx + cy * cy + cz * cz) + 1e-3f, 1.f);
}

// Sample i of the ray: where it meets the sphere of radius n_steps /
// (n_steps - i - 0.5) on the way out (skipped inside the first radius or where
// it misses), 1 / |position|, and the trilinear cell and fractions in
// (longitude, latitude, layer) (render_lerp_kernel_cuvol.cu:403-428).
struct BgSample {
    bool valid;
    float invr;
    int l[3];
    float f[3];
};

__device__ __forceinline__ BgSample bg_sample(const BgView& b, const BgRay& r, int i) {
    BgSample s;
    s.valid = false;
    s.invr = 0.f;
    if (i >= b.n_steps) return s;
    const float rad = static_cast<float>(b.n_steps) / (static_cast<float>(b.n_steps - i) - 0.5f);
    if (rad < r.inner) return s;
    const float det = r.f + 2.f * r.q2a * rad * rad;
    if (det < 0.f) return s;
    const float t = (-r.qb + sqrtf(det)) / r.q2a;
    float p[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) p[j] = fmaf(t, r.d[j], r.o[j]);
    const float invr = 1.0f / sqrtf(bg_dot(p, p));
#pragma unroll
    for (int j = 0; j < 3; ++j) p[j] *= invr;
    // Equirectangular pixel of the unit direction (_unitvec2equirect,
    // render_util.cuh:482-490).
    const float lat = asinf(p[1]);
    const float lon = atan2f(p[0], p[2]);
    const float x = static_cast<float>(2 * b.reso) * (0.5f + lon * (0.5f * kInvPi));
    const float y = static_cast<float>(b.reso) * (0.5f - lat * kInvPi);
    const float z = fminf(fmaxf((1.f - invr) * static_cast<float>(b.nlayers) - 0.5f, 0.f),
                          static_cast<float>(b.nlayers - 1));
    // Truncation toward zero as the reference's (int) casts; the lower clamp
    // only keeps a NaN position (a direction rounded just past a pole) inside.
    s.l[0] = max(min(static_cast<int>(x), 2 * b.reso - 1), 0);
    s.l[1] = max(min(static_cast<int>(y), b.reso - 1), 0);
    s.l[2] = max(min(static_cast<int>(z), b.nlayers - 2), 0);
    s.f[0] = x - static_cast<float>(s.l[0]);
    s.f[1] = y - static_cast<float>(s.l[1]);
    s.f[2] = z - static_cast<float>(s.l[2]);
    s.invr = invr;
    s.valid = true;
    return s;
}

// Row offset (link * nlayers + layer) of pixel column (x, y), or -1.
__device__ __forceinline__ int64_t bg_row(const BgView& b, int x, int y, int l2) {
    const int link = b.links[x * b.reso + y];
    if (link < 0 || link >= b.rows) return -1;
    return static_cast<int64_t>(link) * b.nlayers + l2;
}

__device__ __forceinline__ float4 lerp4(float4 a, float4 c, float w) {
    return make_float4(lerpf(a.x, c.x, w), lerpf(a.y, c.y, w), lerpf(a.z, c.z, w),
                       lerpf(a.w, c.w, w));
}

__device__ __forceinline__ float4 bg_column(const BgView& b, int64_t row, float f2) {
    if (row < 0) return make_float4(0.f, 0.f, 0.f, 0.f);
    return lerp4(b.data[row], b.data[row + 1], f2);
}

// The four pixel columns of a sample: (x, y), (x, ny), (nx, y), (nx, ny),
// wrapping at the image edges (trilerp_bg_one, render_util.cuh:157-189).
struct BgCorners {
    int64_t row[4];
};

__device__ __forceinline__ BgCorners bg_corners(const BgView& b, const BgSample& s) {
    const int ny = s.l[1] < b.reso - 1 ? s.l[1] + 1 : 0;
    const int nx = s.l[0] < 2 * b.reso - 1 ? s.l[0] + 1 : 0;
    BgCorners c;
    c.row[0] = bg_row(b, s.l[0], s.l[1], s.l[2]);
    c.row[1] = bg_row(b, s.l[0], ny, s.l[2]);
    c.row[2] = bg_row(b, nx, s.l[1], s.l[2]);
    c.row[3] = bg_row(b, nx, ny, s.l[2]);
    return c;
}

__device__ __forceinline__ float4 bg_value(const BgView& b, const BgSample& s,
                                           const BgCorners& c) {
    const float4 v00 = bg_column(b, c.row[0], s.f[2]);
    const float4 v01 = bg_column(b, c.row[1], s.f[2]);
    const float4 v10 = bg_column(b, c.row[2], s.f[2]);
    const float4 v11 = bg_column(b, c.row[3], s.f[2]);
    return lerp4(lerp4(v00, v01, s.f[1]), lerp4(v10, v11, s.f[1]), s.f[0]);
}

// 32-lane group helpers (the group is one half of the wavefront; every lane of
// the group is active wherever these are called).
__device__ __forceinline__ uint32_t bg_ballot(bool p) {
    return static_cast<uint32_t>(__ballot(p) >> (threadIdx.x & 32u));
}
// Inclusive prefix sum over the group by DPP moves (no LDS round trips): shifts
// within each 16-lane row, then the group's second row adds the first one's
// total.
template <int CTRL>
__device__ __forceinline__ float bg_dpp(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ float bg_scan(float v) {
    v += bg_dpp<0x111>(v);  // row_shr:1
    v += bg_dpp<0x112>(v);
    v += bg_dpp<0x114>(v);
    v += bg_dpp<0x118>(v);
    // row_bcast:15 into rows 1 and 3
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x142, 0xA, 0xF, false));
    return v;
}
__device__ __forceinline__ float bg_sum(float v) {
#pragma unroll
    for (int m = kBgGroup / 2; m >= 1; m >>= 1) v += __shfl_xor(v, m, kBgGroup);
    return v;
}

// Per-chunk march state shared by the forward and the backward.
struct BgChunk {
    BgSample s;
    BgCorners c;
    float4 v;
    float il;        // 1 / radius of the previous placed sample
    float pcnt;      // optical depth of the sample (0 unless it contributes)
    float lt_after;  // log transmittance after the sample
    float incl;      // inclusive scan of pcnt
    bool live;       // contributes and is not past the stop
    int stop_lane;   // the chunk's last live lane or 31
    bool stopped;
};

// Places and reads chunk `base` of the ray; advances invr_last.  lt is the log
// transmittance before the chunk.
__device__ __forceinline__ void bg_chunk(const BgView& b, const BgRay& r, int base, int lane,
                                         float lt, float& invr_last, BgChunk& k) {
    k.s = bg_sample(b, r, base + lane);
    const uint32_t vm = bg_ballot(k.s.valid);
    const uint32_t below = vm & ((1u << lane) - 1u);
    const int src = below ? 31 - static_cast<int>(__clz(below)) : lane;
    const float prev = __shfl(k.s.invr, src, kBgGroup);
    k.il = below ? prev : invr_last;
    if (vm) invr_last = __shfl(k.s.invr, 31 - static_cast<int>(__clz(vm)), kBgGroup);
    k.v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (k.s.valid) {
        k.c = bg_corners(b, k.s);
        k.v = bg_value(b, k.s, k.c);
    }
    const bool contrib = k.s.valid && k.v.w > 0.f;
    k.pcnt = contrib ? (k.il - k.s.invr) * r.ws * k.v.w : 0.f;
    k.incl = bg_scan(k.pcnt);
    k.lt_after = lt - k.incl;
    const uint32_t stopm = bg_ballot(contrib && __expf(k.lt_after) < b.stop);
    k.stopped = stopm != 0u;
    k.stop_lane = k.stopped ? __ffs(stopm) - 1 : kBgGroup - 1;
    k.live = contrib && lane <= k.stop_lane;
}

__device__ __forceinline__ float pick3f(const float* v, int c) {
    return c == 0 ? v[0] : (c == 1 ? v[1] : v[2]);
}

// Background colour of each ray added to rgb [n][3] (render_background_kernel
// / render_background_image_kernel, render_lerp_kernel_cuvol.cu:775-818); rays
// whose grid log transmittance is below -25 get nothing.  bg_rgb_out (may be
// NULL) receives the added colour.
template <bool IMAGE>
__global__ __launch_bounds__(kBgBlock) void k_background(
        BgView b, const float* __restrict__ origins, const float* __restrict__ dirs,
        svox2_camera_t cam, int64_t n, const float* __restrict__ log_t_fg,
        float* __restrict__ rgb, float* __restrict__ bg_rgb_out) {
    const int64_t ray = (static_cast<int64_t>(blockIdx.x) * kBgBlock + threadIdx.x) / kBgGroup;
    const int lane = threadIdx.x % kBgGroup;
    if (ray >= n) return;
    float lt = log_t_fg[ray];
    if (lt < -25.f) {
        if (bg_rgb_out != nullptr && lane < 3) bg_rgb_out[3 * ray + lane] = 0.f;
        return;
    }
    float wo[3], wd[3];
    if (IMAGE) {
        camera_ray(cam, static_cast<int>(ray % cam.width), static_cast<int>(ray / cam.width), wd,
                   wo);
    } else {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            wo[i] = origins[3 * ray + i];
            wd[i] = dirs[3 * ray + i];
        }
    }
    BgRay r;
    bg_ray(b, wo, wd, r);
    float invr_last = 1.f / r.inner;
    float acc[3] = {0.f, 0.f, 0.f};
    for (int base = 0; base < b.n_steps; base += kBgGroup) {
        BgChunk k;
        bg_chunk(b, r, base, lane, lt, invr_last, k);
        if (k.live) {
            const float w = __expf(k.lt_after + k.pcnt) * (1.f - __expf(-k.pcnt));
            acc[0] += w * fmaxf(fmaf(k.v.x, kShC0, 0.5f), 0.f);
            acc[1] += w * fmaxf(fmaf(k.v.y, kShC0, 0.5f), 0.f);
            acc[2] += w * fmaxf(fmaf(k.v.z, kShC0, 0.5f), 0.f);
        }
        lt -= __shfl(k.incl, k.stop_lane, kBgGroup);
        if (k.stopped) break;
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) acc[c] = bg_sum(acc[c]);
    if (lane < 3) {
        const float val = pick3f(acc, lane) + __expf(lt) * b.bg;
        rgb[3 * ray + lane] += val;
        if (bg_rgb_out != nullptr) bg_rgb_out[3 * ray + lane] = val;
    }
}

// A live sample's gradient terms for the scatter: its four pixel columns in
// slot order (row offset link * nlayers, -1 if empty, and bilinear weight), per
// channel its term, its lower layer and the layer fraction.  Column (dx, dy)
// of the pixel cell with lower corner l takes slot (dx dy) ^ parity(l): the
// columns that two neighbouring cells share keep their slot.
struct __align__(16) BgRec {
    float w[4];
    int at[4];
    float v[4];
    int z;
    float fz;
    int change;  // bit q: column slot q differs from the sample before, 16: the layers move on
    int pad;
};

// The accumulators of one ray's scatter: lane = (layer & 7, channel) holds,
// for each of the four column slots, the gradient of that column at layer
// `layer`, a window of 8 layers of which one column's is 128 contiguous bytes.
// A column is added to memory, one request, when a sample puts another column
// in its slot; a lane's layers when the samples pass on to the next 8.
struct BgScatter {
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    int col[4] = {-1, -1, -1, -1};
    int layer;
    int touched = 0;  // bit q: column slot q at this layer was given a term

    __device__ __forceinline__ void flush(const BgView& b, int q, int ch) {
        if (col[q] >= 0) {
            const int64_t at = static_cast<int64_t>(col[q]) + layer;
            if (acc[q] != 0.f) atomic_add_f32(b.grad + 4 * at + ch, acc[q]);
            if (((touched >> q) & 1) && ch == 0 && b.mask != nullptr) b.mask[at] = 1;
        }
        acc[q] = 0.f;
        touched &= ~(1 << q);
    }
};

// Orders this wavefront's LDS writes before its later LDS reads.
__device__ __forceinline__ void bg_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Background gradients of each ray (render_background_backward_kernel,
// render_lerp_kernel_cuvol.cu:820-860).  dL/drgb is grad_in, or with
// rgb_residual (color_cache - grad_in) * norm (grad_in then holds the
// targets).  The background's own colour is bg_src, or with bg_src_is_fg
// color_cache - bg_src (bg_src then holds the grid's colours); its dot product
// with dL/drgb is the running `accum` the reference carries over from the
// grid's backward.
//
// The atomic requests bound this kernel (about 20 G/s, whatever their width up to
// 64 bytes): added sample by sample, 4 requests of 32 bytes per live sample (34M
// for 65536 rays through 64 layers), it took 1.87 ms.  A ray turns by a fraction
// of a pixel and crosses half a layer per sample, so consecutive samples share
// most of their grid points: kept in registers until the ray leaves a grid point,
// 1.36 ms; until it leaves a column or its 8 layers, so that one instruction adds
// a column's 128 bytes (two requests), 1.25 ms (of which 0.37 ms places and reads
// the samples and 0.10 ms are mask stores: 1.13 ms without a mask).
__global__ __launch_bounds__(kBgBlock) void k_background_backward(
        BgView b, const float* __restrict__ origins, const float* __restrict__ dirs, int64_t n,
        const float* __restrict__ grad_in, const float* __restrict__ color_cache,
        int rgb_residual, float norm, const float* __restrict__ log_t_fg,
        const float* __restrict__ bg_src, int bg_src_is_fg, float sparsity) {
    const int64_t ray = (static_cast<int64_t>(blockIdx.x) * kBgBlock + threadIdx.x) / kBgGroup;
    const int lane = threadIdx.x % kBgGroup;
    if (ray >= n) return;
    float lt = log_t_fg[ray];
    if (lt < -25.f) return;
    float gq[3], bgc[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const float cc = color_cache[3 * ray + c];
        gq[c] = rgb_residual ? (cc - grad_in[3 * ray + c]) * norm : grad_in[3 * ray + c];
        bgc[c] = bg_src_is_fg ? cc - bg_src[3 * ray + c] : bg_src[3 * ray + c];
    }
    float accum = fmaf(bgc[0], gq[0], fmaf(bgc[1], gq[1], bgc[2] * gq[2]));
    float wo[3], wd[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        wo[i] = origins[3 * ray + i];
        wd[i] = dirs[3 * ray + i];
    }
    BgRay r;
    bg_ray(b, wo, wd, r);
    __shared__ BgRec shared[kBgBlock];
    BgRec* recs = shared + (threadIdx.x & ~(kBgGroup - 1));
    const int l8 = lane >> 2, ch = lane & 3;
    BgScatter sc;
    sc.layer = l8;
    int last_z = 0;  // the window of layers 0 .. 7
    float invr_last = 1.f / r.inner;
    for (int base = 0; base < b.n_steps; base += kBgGroup) {
        BgChunk k;
        bg_chunk(b, r, base, lane, lt, invr_last, k);
        float w = 0.f, col[3] = {0.f, 0.f, 0.f}, total = 0.f;
        if (k.live) {
            w = __expf(k.lt_after + k.pcnt) * (1.f - __expf(-k.pcnt));
            col[0] = fmaf(k.v.x, kShC0, 0.5f);
            col[1] = fmaf(k.v.y, kShC0, 0.5f);
            col[2] = fmaf(k.v.z, kShC0, 0.5f);
#pragma unroll
            for (int c = 0; c < 3; ++c) total += fmaxf(col[c], 0.f) * gq[c];
        }
        const float acc_incl = bg_scan(w * total);
        // The live samples' records, compacted in march order.
        const uint32_t live = bg_ballot(k.live);
        if (k.live) {
            BgRec& R = recs[__popc(live & ((1u << lane) - 1u))];
#pragma unroll
            for (int c = 0; c < 3; ++c) R.v[c] = col[c] > 0.f ? kShC0 * w * gq[c] : 0.f;
            const float accum_after = accum - acc_incl;
            float gs = r.ws * (k.il - k.s.invr) * (total * __expf(k.lt_after) - accum_after);
            if (sparsity > 0.f)
                gs += sparsity * (4.f * k.v.w / (1.f + 2.f * (k.v.w * k.v.w)));
            R.v[3] = gs;
            const int parity = ((k.s.l[0] & 1) << 1) | (k.s.l[1] & 1);
            const float ax = 1.f - k.s.f[0], ay = 1.f - k.s.f[1];
#pragma unroll
            for (int q = 0; q < 4; ++q) {  // column: bits dx dy
                const int64_t row = k.c.row[q];
                R.w[q ^ parity] = ((q & 1) ? k.s.f[1] : ay) * ((q & 2) ? k.s.f[0] : ax);
                R.at[q ^ parity] = row < 0 ? -1 : static_cast<int>(row) - k.s.l[2];
            }
            R.z = k.s.l[2];
            R.fz = k.s.f[2];
        }
        bg_lds_fence();
        const int n_live = __popc(live);
        if (n_live > 0) {
            // What each sample changes, found by a lane per sample: the loop
            // below then branches on one word.
            if (lane < n_live) {
                const BgRec& P = recs[max(lane - 1, 0)];
                const int4 pc = *reinterpret_cast<const int4*>(P.at);
                const int4 cc = *reinterpret_cast<const int4*>(recs[lane].at);
                const bool first = lane == 0;
                const int zp = first ? last_z : P.z, zc = recs[lane].z;
                int change = ((first ? sc.col[0] : pc.x) != cc.x ? 1 : 0) |
                             ((first ? sc.col[1] : pc.y) != cc.y ? 2 : 0) |
                             ((first ? sc.col[2] : pc.z) != cc.z ? 4 : 0) |
                             ((first ? sc.col[3] : pc.w) != cc.w ? 8 : 0);
                if ((zp + 1) >> 3 != (zc + 1) >> 3 || ((zp & 7) == 7) != ((zc & 7) == 7))
                    change |= 16;
                recs[lane].change = change;
            }
            bg_lds_fence();
            float4 w4 = *reinterpret_cast<const float4*>(recs[0].w);
            int4 z4 = *reinterpret_cast<const int4*>(&recs[0].z);
            float vc = recs[0].v[ch];
            for (int j = 0; j < n_live; ++j) {
                const BgRec& N = recs[min(j + 1, n_live - 1)];  // on its way for the next turn
                const float4 w4n = *reinterpret_cast<const float4*>(N.w);
                const int4 z4n = *reinterpret_cast<const int4*>(&N.z);
                const float vcn = N.v[ch];
                const int z = z4.x;
                const float fz = __int_as_float(z4.y);
                // The lane's layer: the one of its 8 that the sample's upper
                // layer is among, except that the lower layer keeps its lane.
                const bool lower = (z & 7) == l8, upper = ((z + 1) & 7) == l8;
                if (z4.z != 0) {
                    const int layer = lower ? z : ((z + 1) & ~7) + l8;
                    const int4 c4 = *reinterpret_cast<const int4*>(recs[j].at);
                    const int cq[4] = {c4.x, c4.y, c4.z, c4.w};
                    const bool moved = layer != sc.layer;
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        if (moved || ((z4.z >> q) & 1)) sc.flush(b, q, ch);
                        sc.col[q] = cq[q];
                    }
                    sc.layer = layer;
                }
                const float t = lower ? vc * (1.f - fz) : (upper ? vc * fz : 0.f);
                sc.acc[0] = fmaf(w4.x, t, sc.acc[0]);
                sc.acc[1] = fmaf(w4.y, t, sc.acc[1]);
                sc.acc[2] = fmaf(w4.z, t, sc.acc[2]);
                sc.acc[3] = fmaf(w4.w, t, sc.acc[3]);
                if (lower || upper) sc.touched = 15;
                last_z = z;
                w4 = w4n;
                z4 = z4n;
                vc = vcn;
            }
        }
        bg_lds_fence();  // the records are rewritten by the next chunk
        lt -= __shfl(k.incl, k.stop_lane, kBgGroup);
        accum -= __shfl(acc_incl, k.stop_lane, kBgGroup);
        if (k.stopped) break;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) sc.flush(b, q, ch);
}

// Total variation of an MSI (msi_tv_grad_sparse_kernel,
// loss_kernel.cu:248-333): one thread per listed cell, all its channels.
__global__ __launch_bounds__(256) void k_msi_tv(const int32_t* __restrict__ links, int reso,
                                                const float* __restrict__ msi, int64_t rows,
                                                int nl, int nc,
                                                const int32_t* __restrict__ cells, int64_t n,
                                                float scale, float scale_last,
                                                uint8_t* __restrict__ mask,
                                                float* __restrict__ grad) {
    const int64_t tid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (tid >= n) return;
    const int idx = cells[tid];
    const int64_t total = static_cast<int64_t>(2 * reso) * reso * nl;
    if (idx < 0 || idx >= total) return;
    const int z = idx % nl;
    const int tmp = idx / nl;
    const int y = tmp % reso;
    const int x = tmp / reso;
    const int nx = x == 2 * reso - 1 ? 0 : x + 1;
    const int ny = y == reso - 1 ? 0 : y + 1;
    auto link_of = [&](int xx, int yy) {
        const int l = links[xx * reso + yy];
        return (l >= 0 && l < rows) ? l : -1;
    };
    const int l00 = link_of(x, y), l01 = link_of(x, ny), l10 = link_of(nx, y);
    const float fx = static_cast<float>(2 * reso) * (1.f / 256.f);
    const float fy = static_cast<float>(reso) * (1.f / 256.f);
    const float fz = static_cast<float>(nl) * (1.f / 256.f);
    auto val = [&](int l, int zz, int c) {
        return msi[(static_cast<int64_t>(l) * nl + zz) * nc + c];
    };
    auto add = [&](int l, int zz, int c, float v, float idelta) {
        if (l < 0 || v == 0.f) return;
        const int64_t r = static_cast<int64_t>(l) * nl + zz;
        atomic_add_f32(grad + r * nc + c, v * idelta);
        if (mask != nullptr) mask[r] = 1;
    };
    for (int c = 0; c < nc; ++c) {
        const bool last = c == nc - 1;
        const float v00 = l00 >= 0 ? val(l00, z, c) : 0.f;
        const float vz = (l00 >= 0 && z + 1 < nl) ? val(l00, z + 1, c) : (last ? 0.f : v00);
        const float v01 = l01 >= 0 ? val(l01, z, c) : 0.f;
        const float v10 = l10 >= 0 ? val(l10, z, c) : 0.f;
        float dx = v10 - v00, dy = v01 - v00, dz = vz - v00;
        const float idelta = (last ? scale_last : scale) * rsqrtf(1e-9f + dx * dx + dy * dy + dz * dz);
        dx *= fx;
        dy *= fy;
        dz *= fz;
        add(l00, z, c, -(dx + dy + dz), idelta);
        if (z + 1 < nl) add(l00, z + 1, c, dz, idelta);
        add(l01, z, c, dy, idelta);
        add(l10, z, c, dx, idelta);
    }
}

int make_bg_view(const svox2_grid_t* g, float step, float bg, float stop, BgView& b) {
    SVOX2_REQUIRE(g->background_data != nullptr, "grid.background_data is NULL");
    SVOX2_REQUIRE(g->background_reso >= 1 && g->background_reso < 32768,
                  "background_reso %d out of range", g->background_reso);
    SVOX2_REQUIRE(g->background_nlayers >= 2, "background_nlayers %d must be >= 2",
                  g->background_nlayers);
    SVOX2_REQUIRE(g->background_rows >= 0 &&
                      g->background_rows * g->background_nlayers < INT_MAX,
                  "background_rows %lld x nlayers %d exceeds int32 layer indices",
                  (long long)g->background_rows, g->background_nlayers);
    SVOX2_REQUIRE(reinterpret_cast<uintptr_t>(g->background_data) % 16 == 0,
                  "background_data must be 16-byte aligned");
    SVOX2_REQUIRE(step > 0.f, "step_size must be > 0");
    const float steps = static_cast<float>(g->background_nlayers) / step;
    SVOX2_REQUIRE(steps < 1e6f, "background needs too many steps (%g)", (double)steps);
    b.links = g->background_links;
    b.data = reinterpret_cast<const float4*>(g->background_data);
    b.grad = nullptr;
    b.mask = nullptr;
    b.rows = g->background_rows;
    b.reso = g->background_reso;
    b.nlayers = g->background_nlayers;
    b.n_steps = static_cast<int>(steps) + 2;
    for (int i = 0; i < 3; ++i) {
        b.offset[i] = g->offset[i];
        b.scaling[i] = g->scaling[i];
        b.sph[i] = 2.f / static_cast<float>(g->size[i]);
    }
    b.bg = bg;
    b.stop = stop;
    return ok();
}

}  // namespace

bool grid_has_background(const svox2_grid_t* g) {
    return g != nullptr && g->background_links != nullptr && g->background_nlayers > 0;
}

int check_background(const svox2_grid_t* g, const svox2_render_options_t* opt) {
    BgView b;
    return make_bg_view(g, opt->step_size, opt->background_brightness, opt->stop_thresh, b);
}

int launch_background(const svox2_grid_t* g, const svox2_render_options_t* opt,
                      const float* origins, const float* dirs, const svox2_camera_t* cam,
                      int64_t n, const float* log_t_fg, float* rgb, float* bg_rgb_out,
                      hipStream_t s) {
    BgView b;
    int st = make_bg_view(g, opt->step_size, opt->background_brightness, opt->stop_thresh, b);
    if (st) return st;
    if (n == 0) return ok();
    const unsigned blocks = blocks_for(n * kBgGroup, kBgBlock);
    if (cam != nullptr)
        hipLaunchKernelGGL(k_background<true>, dim3(blocks), dim3(kBgBlock), 0, s, b, origins,
                           dirs, *cam, n, log_t_fg, rgb, bg_rgb_out);
    else
        hipLaunchKernelGGL(k_background<false>, dim3(blocks), dim3(kBgBlock), 0, s, b, origins,
                           dirs, svox2_camera_t{}, n, log_t_fg, rgb, bg_rgb_out);
    return check_launch("background");
}

int launch_background_backward(const svox2_grid_t* g, const svox2_render_options_t* opt,
                               const float* origins, const float* dirs, int64_t n,
                               const float* grad_in, const float* color_cache, int rgb_residual,
                               float norm, const float* log_t_fg, const float* bg_src,
                               int bg_src_is_fg, float sparsity, const svox2_grads_t* grads,
                               hipStream_t s) {
    BgView b;
    int st = make_bg_view(g, opt->step_size, opt->background_brightness, opt->stop_thresh, b);
    if (st) return st;
    if (grads == nullptr || grads->grad_background_out == nullptr || n == 0) return ok();
    b.grad = grads->grad_background_out;
    b.mask = grads->mask_background_out;
    const unsigned blocks = blocks_for(n * kBgGroup, kBgBlock);
    hipLaunchKernelGGL(k_background_backward, dim3(blocks), dim3(kBgBlock), 0, s, b, origins,
                       dirs, n, grad_in, color_cache, rgb_residual, norm, log_t_fg, bg_src,
                       bg_src_is_fg, sparsity);
    return check_launch("background backward");
}

}  // namespace svox2amd

using namespace svox2amd;

extern "C" int svox2_msi_tv_grad_sparse(const int32_t* links, int32_t reso, const float* msi,
                                        int64_t msi_rows, int32_t nlayers, int32_t nchannels,
                                        const int32_t* rand_cells, int64_t n_cells,
                                        uint8_t* mask_out, float scale, float scale_last,
                                        float* grad_msi, void* stream) {
    SVOX2_REQUIRE(reso >= 1 && reso < 32768, "reso %d out of range", reso);
    SVOX2_REQUIRE(nlayers >= 1 && nchannels >= 1, "nlayers / nchannels must be >= 1");
    SVOX2_REQUIRE(msi_rows >= 0 && msi_rows < INT_MAX, "msi_rows out of range");
    SVOX2_REQUIRE(static_cast<int64_t>(2 * reso) * reso * nlayers < INT_MAX,
                  "MSI has too many cells for int32 indices");
    SVOX2_REQUIRE(n_cells >= 0, "negative cell count");
    if (n_cells == 0) return ok();
    SVOX2_REQUIRE(links != nullptr && rand_cells != nullptr && grad_msi != nullptr &&
                      (msi != nullptr || msi_rows == 0),
                  "links / msi / rand_cells / grad_msi are NULL");
    const float nl = static_cast<float>(n_cells);
    hipLaunchKernelGGL(k_msi_tv, dim3(blocks_for(n_cells, 256)), dim3(256), 0,
                       static_cast<hipStream_t>(stream), links, reso, msi, msi_rows, nlayers,
                       nchannels, rand_cells, n_cells, scale / nl, scale_last / nl, mask_out,
                       grad_msi);
    return check_launch("msi_tv_grad_sparse");
}
