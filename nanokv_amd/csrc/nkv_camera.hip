// nkv_camera.hip -- camera PRoPE transform of bf16 rows (nkv_camera_apply) and
// the validation of nkv_camera shared with nkv_attend.
//
// Each 4-vector of a row is multiplied by the sub-frame matrix of the row's
// frame (nkv_camera.h).
#include "nkv_camera.h"

#include "nkv_internal.h"

#include <type_traits>

namespace nkv {

int camera_from_abi(const nkv_camera* c, int D, int B, CameraDev* dev) {
    NKV_REQUIRE(c, NKV_ERR_INVALID, "camera is null");
    NKV_REQUIRE(c->mats && c->frame_mat, NKV_ERR_INVALID, "camera needs mats and frame_mat");
    NKV_REQUIRE(c->n_mats >= 1 && c->n_frames >= 1 && c->tokens_per_frame >= 1 && c->mats_bs >= 0,
                NKV_ERR_INVALID, "camera needs n_mats, n_frames, tokens_per_frame >= 1");
    NKV_REQUIRE(((uintptr_t)c->mats & 15) == 0 && c->mats_bs % 4 == 0, NKV_ERR_INVALID,
                "camera mats must be 16-byte aligned (mats_bs a multiple of 4)");
    NKV_REQUIRE(c->layout == NKV_CAMERA_FULL || c->layout == NKV_CAMERA_SF13, NKV_ERR_INVALID,
                "unknown camera layout");
    NKV_REQUIRE(c->layout != NKV_CAMERA_FULL || (D > 0 && D % 64 == 0), NKV_ERR_INVALID,
                "the FULL camera layout needs D % 64 == 0");
    NKV_REQUIRE(c->layout != NKV_CAMERA_SF13 || D >= 32, NKV_ERR_INVALID,
                "the SF13 camera layout needs D >= 32");
    NKV_REQUIRE(c->mats_bs == 0 || B <= c->n_batches, NKV_ERR_INVALID,
                "camera mats hold fewer matrix batches than the call's batch items");
    dev->mats = c->mats;
    dev->mats_bs = c->mats_bs;
    dev->n_mats = c->n_mats;
    dev->layout = c->layout;
    dev->frame_mat = c->frame_mat;
    dev->n_frames = c->n_frames;
    dev->tokens_per_frame = c->tokens_per_frame;
    dev->blocks = nullptr;
    return NKV_OK;
}

namespace {

struct CameraApplyParams {
    CameraDev cam;
    int B, H, D;
    int64_t S;
    const uint16_t* x;
    int64_t x_sb, x_st, x_sh;
    const int32_t* rows;
    uint16_t* out;
    int64_t o_sb, o_st, o_sh;
};

__global__ void __launch_bounds__(256) camera_apply_kernel(CameraApplyParams p) {
    const int nv = camera_vectors(p.cam.layout, p.D);
    const int64_t total = (int64_t)p.B * p.S * p.H * nv;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int v = (int)(i % nv);
        int64_t rest = i / nv;
        const int h = (int)(rest % p.H);
        rest /= p.H;
        const int64_t s = rest % p.S;
        const int b = (int)(rest / p.S);
        const int64_t row = p.rows ? (int64_t)p.rows[s] : s;
        int base, step, sub;
        camera_vector_dims(p.cam.layout, p.D, v, base, step, sub);
        const uint16_t* src = p.x + b * p.x_sb + s * p.x_st + h * p.x_sh + base;
        uint16_t* dst = p.out + b * p.o_sb + s * p.o_st + h * p.o_sh + base;
        if (sub < 0) {  // dims the layout leaves alone
#pragma unroll
            for (int j = 0; j < 4; ++j) dst[j * step] = src[j * step];
            continue;
        }
        float x[4], y[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = bf16_bits_to_f32(src[j * step]);
        camera_vec4(camera_mats(p.cam, b, row) + 16 * sub, x, y);
#pragma unroll
        for (int j = 0; j < 4; ++j) dst[j * step] = f32_to_bf16_bits(y[j]);
    }
}

// 16-byte pieces: one thread transforms piece `part` (8 dims, two 4-vectors)
// of one (b, s) in HEADS heads: the frame's matrices are fetched and rounded
// once for them, their loads are in flight together.
// INTER: the vectors are the even and the odd dims, one sub-frame (FULL at
// D = 128); else dims 0..3 and 4..7, each with its own sub-frame or (< 0) left
// alone (FULL at D = 64, SF13).  Per call in a graph with 1, 2, 4, 8 and 16
// heads, FULL, us: 37 x 8 x 128 2.57, 2.82, 3.31, 4.34, 7.2 (a thread's chain over
// its heads); 780 x 24 4.48, 4.27, 4.34, 4.96, 13.1; 1,560 x 24 (19 MB moved)
// 6.74, 5.85, 5.72, 6.50, 15.5; 3,120 x 24 10.6, 9.3, 8.6, 9.4; 12,480 x 24 31.0,
// 30.6, 29.7, 30.6 (SF13 38.6, 32.2, 28.1, 26.1); one 4-vector per thread, four
// 2-byte accesses each way: 2.82, 7.60, 12.2, 21.0, 72.  Two up to PIECES_FEW
// pieces, eight above.
constexpr int64_t PIECES_FEW = 512 << 10;

template <bool INTER, int CA_HEADS>
__global__ void __launch_bounds__(256) camera_pieces_kernel(CameraApplyParams p, uint32_t items) {
    const uint32_t per_row = (uint32_t)p.D / 8, S = (uint32_t)p.S;
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= items) return;
    const uint32_t bs = i / per_row, part = i - bs * per_row, b = bs / S, s = bs - b * S;
    const int h0 = blockIdx.y * CA_HEADS;
    const uint16_t* src = p.x + b * p.x_sb + s * p.x_st + h0 * p.x_sh + 8 * part;
    uint16_t* dst = p.out + b * p.o_sb + s * p.o_st + h0 * p.o_sh + 8 * part;
    u32x4 w[CA_HEADS];
#pragma unroll
    for (int h = 0; h < CA_HEADS; ++h)
        if (h0 + h < p.H) w[h] = *reinterpret_cast<const u32x4*>(src + h * p.x_sh);
    const float* mats = camera_mats(p.cam, (int)b, p.rows ? (int64_t)p.rows[s] : (int64_t)s);
    double m[16];
    auto matrix = [&](int sub) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float4 f = reinterpret_cast<const float4*>(mats + 16 * sub)[q];
            m[4 * q] = (double)bf16_round(f.x);
            m[4 * q + 1] = (double)bf16_round(f.y);
            m[4 * q + 2] = (double)bf16_round(f.z);
            m[4 * q + 3] = (double)bf16_round(f.w);
        }
    };
    auto lo = [](uint32_t x) { return __uint_as_float(x << 16); };
    auto hi = [](uint32_t x) { return __uint_as_float(x & 0xffff0000u); };
    if constexpr (INTER) {
        matrix(part & 3);
#pragma unroll
        for (int h = 0; h < CA_HEADS; ++h) {
            if (h0 + h >= p.H) break;
            float a[4], c[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) { a[j] = lo(w[h][j]); c[j] = hi(w[h][j]); }
#pragma unroll
            for (int r = 0; r < 4; ++r)
                w[h][r] = pack_bf16x2(camera_dot(m + 4 * r, a), camera_dot(m + 4 * r, c));
        }
    } else {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            int base, step, sub;
            camera_vector_dims(p.cam.layout, p.D, 2 * (int)part + u, base, step, sub);
            if (sub < 0) continue;
            matrix(sub);
#pragma unroll
            for (int h = 0; h < CA_HEADS; ++h) {
                if (h0 + h >= p.H) break;
                const float a[4] = {lo(w[h][2 * u]), hi(w[h][2 * u]), lo(w[h][2 * u + 1]),
                                    hi(w[h][2 * u + 1])};
                w[h][2 * u] = pack_bf16x2(camera_dot(m, a), camera_dot(m + 4, a));
                w[h][2 * u + 1] = pack_bf16x2(camera_dot(m + 8, a), camera_dot(m + 12, a));
            }
        }
    }
#pragma unroll
    for (int h = 0; h < CA_HEADS; ++h)
        if (h0 + h < p.H) *reinterpret_cast<u32x4*>(dst + h * p.o_sh) = w[h];
}

// The 16-byte kernel where rows are whole aligned pieces and a piece's two
// vectors lie in it; one 4-vector per thread for the rest (FULL at D >= 192,
// odd strides).
int camera_launch(hipStream_t s, const CameraApplyParams& p) {
    const int D = p.D, layout = p.cam.layout;
    const int64_t pieces = (int64_t)p.B * p.S * (D / 8);
    const bool fits = layout == NKV_CAMERA_SF13 || D == 64 || D == 128;
    if (D % 8 == 0 && fits && pieces <= INT32_MAX && cdiv(p.H, 8) <= 65535 &&
        rows16(p.x, p.x_sb, p.x_st, p.x_sh) && rows16(p.out, p.o_sb, p.o_st, p.o_sh)) {
        auto run = [&](auto inter, auto heads) {
            const dim3 grid((unsigned)cdiv(pieces, 256), (unsigned)cdiv(p.H, heads()));
            camera_pieces_kernel<inter(), heads()><<<grid, 256, 0, s>>>(p, (uint32_t)pieces);
        };
        auto split = [&](auto heads) {
            if (layout == NKV_CAMERA_FULL && D == 128) run(std::true_type{}, heads);
            else run(std::false_type{}, heads);
        };
        if (pieces * p.H <= PIECES_FEW && cdiv(p.H, 2) <= 65535) split(std::integral_constant<int, 2>{});
        else split(std::integral_constant<int, 8>{});
    } else {
        const int64_t items = (int64_t)p.B * p.S * p.H * camera_vectors(layout, D);
        const unsigned grid = (unsigned)std::min<int64_t>(cdiv(items, 256), 65536);
        camera_apply_kernel<<<grid, 256, 0, s>>>(p);
    }
    NKV_LAUNCH_CHECK();
    return NKV_OK;
}

}  // namespace
}  // namespace nkv

using namespace nkv;

namespace nkv {

int camera_apply_inplace(hipStream_t s, const CameraDev& cam, int B, int64_t S, int H, int D,
                         uint16_t* x, int64_t sb, int64_t st, int64_t sh) {
    if ((int64_t)B * S * H == 0) return NKV_OK;
    CameraApplyParams p;
    p.cam = cam;
    p.B = B;
    p.H = H;
    p.D = D;
    p.S = S;
    p.x = x;
    p.x_sb = sb;
    p.x_st = st;
    p.x_sh = sh;
    p.rows = nullptr;
    p.out = x;
    p.o_sb = sb;
    p.o_st = st;
    p.o_sh = sh;
    return camera_launch(s, p);
}

}  // namespace nkv

extern "C" int nkv_camera_apply(void* stream, const nkv_camera* camera, int B, int64_t S, int H,
                                int D, const uint16_t* x, int64_t x_sb, int64_t x_st,
                                int64_t x_sh, const int32_t* rows, uint16_t* out, int64_t o_sb,
                                int64_t o_st, int64_t o_sh) {
    clear_error();
    CameraApplyParams p;
    int rc = camera_from_abi(camera, D, B, &p.cam);
    if (rc) return rc;
    NKV_REQUIRE(B >= 0 && S >= 0 && H >= 0, NKV_ERR_INVALID, "negative shape");
    if ((int64_t)B * S * H == 0) return NKV_OK;
    NKV_REQUIRE(x && out, NKV_ERR_INVALID, "x and out are required");
    NKV_REQUIRE(D % 4 == 0, NKV_ERR_INVALID, "D must be a multiple of 4");
    p.B = B;
    p.H = H;
    p.D = D;
    p.S = S;
    p.x = x;
    p.x_sb = x_sb;
    p.x_st = x_st;
    p.x_sh = x_sh;
    p.rows = rows;
    p.out = out;
    p.o_sb = o_sb;
    p.o_st = o_st;
    p.o_sh = o_sh;
    return camera_launch((hipStream_t)stream, p);
}
