// nkv_rope.hip -- RoPE of bf16 rows at codec-row positions (nkv_rope_apply)
// and the validation of nkv_rope shared with nkv_attend.
//
// Restates rope_apply (wan_video_dit.py:185-192): x in fp64, times the
// position's complex frequency, cast to bf16; the frequency of pair p comes
// from one of three bands (nkv_rope.h).  Memory-bound.
#include "nkv_rope.h"

#include "nkv_internal.h"

namespace nkv {

int rope_from_abi(const nkv_rope* r, int D, RopeDev* dev) {
    NKV_REQUIRE(r, NKV_ERR_INVALID, "rope is null");
    NKV_REQUIRE(D > 0 && D % 2 == 0, NKV_ERR_INVALID, "RoPE needs an even head dimension");
    if (r->cs_rows) {
        NKV_REQUIRE(r->n_rows >= 1, NKV_ERR_INVALID, "a per-row RoPE table needs n_rows >= 1");
        *dev = RopeDev{};
        dev->cs_rows = r->cs_rows;
        dev->n_rows = r->n_rows;
        dev->pt = D / 2;
        return NKV_OK;
    }
    NKV_REQUIRE(r->pt >= 0 && r->ph >= 0 && r->pw >= 0 && r->pt + r->ph + r->pw == D / 2,
                NKV_ERR_INVALID, "RoPE bands must hold D / 2 pairs (pt + ph + pw)");
    NKV_REQUIRE(r->grid_h >= 1 && r->grid_w >= 1 && r->n_frames >= 1, NKV_ERR_INVALID,
                "RoPE needs grid_h, grid_w and n_frames >= 1");
    NKV_REQUIRE(r->pt == 0 || (r->cs_t && r->frame_pos && r->n_t >= 1), NKV_ERR_INVALID,
                "RoPE temporal band needs cs_t, frame_pos and n_t >= 1");
    NKV_REQUIRE(r->ph == 0 || r->cs_h, NKV_ERR_INVALID, "RoPE row band needs cs_h");
    NKV_REQUIRE(r->n_frames * (int64_t)r->grid_h * r->grid_w < INT32_MAX, NKV_ERR_INVALID,
                "RoPE frames must cover fewer than 2^31 rows");
    NKV_REQUIRE(r->pw == 0 || r->cs_w, NKV_ERR_INVALID, "RoPE column band needs cs_w");
    dev->cs_t = r->cs_t;
    dev->cs_h = r->cs_h;
    dev->cs_w = r->cs_w;
    dev->frame_pos = r->frame_pos;
    dev->n_frames = r->n_frames;
    dev->n_t = r->n_t;
    dev->pt = r->pt;
    dev->ph = r->ph;
    dev->pw = r->pw;
    dev->grid_h = r->grid_h;
    dev->grid_w = r->grid_w;
    dev->pairs = nullptr;
    return NKV_OK;
}

namespace {

struct RopeApplyParams {
    RopeDev rope;
    int B, H, D;
    int64_t S;
    const uint16_t* x;
    int64_t x_sb, x_st, x_sh;
    const int32_t* rows;
    uint16_t* out;
    int64_t o_sb, o_st, o_sh;
};

// 16-byte pieces (D % 8 == 0): one thread rotates the four pairs of piece
// `part` of one (b, s) in HEADS heads, so that the position's index arithmetic
// and its four (cos, sin) entries are fetched once for them and their loads are
// in flight together (one head per thread took four 64-bit divisions and 64
// bytes of table per 16 of x).  Per call in a graph with 1, 2, 4, 8 and 16 heads,
// a table per row, us: 37 x 8 x 128 2.25, 2.35, 2.61, 3.14, 5.6 (a thread's chain
// over its heads); 780 x 24 4.05, 3.59, 3.60, 3.80, 10.3; 1,560 x 24 (19 MB
// moved) 6.05, 4.99, 4.99, 5.29, 13.8; 2,340 x 24 10.0, 8.25, 7.55, 6.58; 12,480
// x 24 47.9, 42.0, 34.0, 28.9 (the table's traffic).  Two up to PIECES_FEW
// pieces, eight above.
constexpr int64_t PIECES_FEW = 512 << 10;

template <int RA_HEADS>
__global__ void __launch_bounds__(256) rope_pieces_kernel(RopeApplyParams p, uint32_t items) {
    const uint32_t per_row = (uint32_t)p.D / 8, S = (uint32_t)p.S;
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= items) return;
    const uint32_t bs = i / per_row, part = i - bs * per_row, b = bs / S, s = bs - b * S;
    const int h0 = blockIdx.y * RA_HEADS;
    const uint16_t* src = p.x + b * p.x_sb + s * p.x_st + h0 * p.x_sh + 8 * part;
    uint16_t* dst = p.out + b * p.o_sb + s * p.o_st + h0 * p.o_sh + 8 * part;
    u32x4 w[RA_HEADS];
#pragma unroll
    for (int h = 0; h < RA_HEADS; ++h)
        if (h0 + h < p.H) w[h] = *reinterpret_cast<const u32x4*>(src + h * p.x_sh);
    const RopeRows rr = rope_rows(p.rope, p.rows ? (int64_t)p.rows[s] : (int64_t)s);
    double c[4], sn[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const f64x2 cs = *reinterpret_cast<const f64x2*>(rope_entry(p.rope, rr, 4 * part + e));
        c[e] = cs[0];
        sn[e] = cs[1];
    }
#pragma unroll
    for (int h = 0; h < RA_HEADS; ++h) {
        if (h0 + h >= p.H) break;
        u32x4 y;
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = rope_pair(w[h][e], c[e], sn[e]);
        *reinterpret_cast<u32x4*>(dst + h * p.o_sh) = y;
    }
}

// One pair per thread: any even D and any strides of whole pairs.
__global__ void __launch_bounds__(256) rope_apply_kernel(RopeApplyParams p) {
    const int per_row = p.D / 2;
    const int64_t total = (int64_t)p.B * p.S * p.H * per_row;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int part = (int)(i % per_row);
        int64_t rest = i / per_row;
        const int h = (int)(rest % p.H);
        rest /= p.H;
        const int64_t s = rest % p.S;
        const int b = (int)(rest / p.S);
        const RopeRows rr = rope_rows(p.rope, p.rows ? (int64_t)p.rows[s] : s);
        const uint16_t* src = p.x + b * p.x_sb + s * p.x_st + h * p.x_sh + 2 * part;
        uint16_t* dst = p.out + b * p.o_sb + s * p.o_st + h * p.o_sh + 2 * part;
        const uint32_t w = *reinterpret_cast<const uint32_t*>(src);
        const double* cs = rope_entry(p.rope, rr, part);
        *reinterpret_cast<uint32_t*>(dst) = rope_pair(w, cs[0], cs[1]);
    }
}

}  // namespace
}  // namespace nkv

using namespace nkv;

extern "C" int nkv_rope_apply(void* stream, const nkv_rope* rope, int B, int64_t S, int H, int D,
                              const uint16_t* x, int64_t x_sb, int64_t x_st, int64_t x_sh,
                              const int32_t* rows, uint16_t* out, int64_t o_sb, int64_t o_st,
                              int64_t o_sh) {
    clear_error();
    RopeApplyParams p;
    int rc = rope_from_abi(rope, D, &p.rope);
    if (rc) return rc;
    NKV_REQUIRE(B >= 0 && S >= 0 && H >= 0, NKV_ERR_INVALID, "negative shape");
    if ((int64_t)B * S * H == 0) return NKV_OK;
    NKV_REQUIRE(x && out, NKV_ERR_INVALID, "x and out are required");
    NKV_REQUIRE(rows || S <= rope_rows_covered(rope), NKV_ERR_INVALID,
                "more rows than the RoPE frames cover");
    NKV_REQUIRE(S < INT32_MAX, NKV_ERR_INVALID, "RoPE rows must fit in 32 bits");
    const bool vec = D % 8 == 0 && (reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(out)) % 16 == 0 &&
                     x_sb % 8 == 0 && x_st % 8 == 0 && x_sh % 8 == 0 && o_sb % 8 == 0 &&
                     o_st % 8 == 0 && o_sh % 8 == 0;
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
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const int64_t pieces = (int64_t)B * S * (D / 8);
    if (vec && pieces <= INT32_MAX && cdiv(H, 8) <= 65535) {
        auto grid = [&](int heads) {
            return dim3((unsigned)cdiv(pieces, 256), (unsigned)cdiv(H, heads));
        };
        if (pieces * H <= PIECES_FEW && cdiv(H, 2) <= 65535)
            rope_pieces_kernel<2><<<grid(2), 256, 0, s>>>(p, (uint32_t)pieces);
        else
            rope_pieces_kernel<8><<<grid(8), 256, 0, s>>>(p, (uint32_t)pieces);
    } else {
        const int64_t items = (int64_t)B * S * H * (D / 2);
        rope_apply_kernel<<<(unsigned)std::min<int64_t>(cdiv(items, 256), 65536), 256, 0, s>>>(p);
    }
    NKV_LAUNCH_CHECK();
    return NKV_OK;
}
