// nkv_merge.hip -- output merges of the Fast partitions of the HY and
// LingBot backbones (gfx950): HY's value lift of its two history branches
// fused with the LSE merge into the native output (nkv_lift_lse_combine), and
// LingBot's finish of one reader group with its value-mean correction and
// head scatter (nkv_finish).  Both are bandwidth-bound epilogues: each output
// element is read once from every input and written once.  Compiled without
// FMA contraction, as the reference kernels are (enable_fp_fusion=False).
#include "nkv_common.h"
#include "nkv_internal.h"

namespace nkv {

namespace {

// ---- nkv_lift_lse_combine (HYP:883-1014)
// One block per (32 queries, batch item b of 2B, head h).  The block's low
// rows and the head's lift (Main [low_dim, 128], or PRoPE mix [low_dim/4, 32])
// are staged in LDS as fp32; thread t computes output column t % 128 of
// queries t / 128, t / 128 + 2, ...  Each output is a sum of bf16 products
// in fp32 (the lift of one low row), merged with the native value by the two
// LSEs.
constexpr int LC_Q = 32;
constexpr int LC_THREADS = 256;
constexpr int LC_MAXK = 96;

__global__ void __launch_bounds__(LC_THREADS) lift_combine_kernel(nkv_lift_combine_args a) {
    __shared__ float low[LC_Q][LC_MAXK + 1];
    __shared__ float w[LC_MAXK * 128];
    const int t = threadIdx.x;
    const int64_t q0 = (int64_t)blockIdx.x * LC_Q;
    const int b = (int)(blockIdx.y / a.H), h = (int)(blockIdx.y % a.H);
    const bool prope = b >= a.B;
    const int K = a.low_dim;
    for (int i = t; i < LC_Q * K; i += LC_THREADS) {
        const int q = i / K, k = i % K;
        const int64_t qi = q0 + q;
        low[q][k] = qi < a.Q ? bf16_bits_to_f32(a.low[b * a.l_sb + h * a.l_sh + qi * a.l_sq +
                                                      k * a.l_sd])
                             : 0.0f;
    }
    if (!prope) {
        for (int i = t; i < K * 128; i += LC_THREADS) {
            const int k = i >> 7, o = i & 127;
            w[i] = bf16_bits_to_f32(a.main_lift[h * a.ml_sh + k * a.ml_sk + o * a.ml_so]);
        }
    } else {
        for (int i = t; i < (K / 4) * 32; i += LC_THREADS) {
            const int k = i >> 5, j = i & 31;
            w[i] = bf16_bits_to_f32(a.prope_mix[h * a.pm_sh + k * a.pm_sk + j * a.pm_so]);
        }
    }
    __syncthreads();
    const int o = t & 127;
    for (int q = t >> 7; q < LC_Q; q += LC_THREADS / 128) {
        const int64_t qi = q0 + q;
        if (qi >= a.Q) break;
        float acc = 0.0f;
        if (!prope) {
            for (int k = 0; k < K; ++k) acc += low[q][k] * w[k * 128 + o];
        } else {
            // output dim 4 j + c of coordinate c takes quartets k of low dim 4 k + c
            const int c = o & 3, j = o >> 2;
            for (int k = 0; k < K / 4; ++k) acc += low[q][4 * k + c] * w[k * 32 + j];
        }
        const float x = a.native_lse[b * a.nl_sb + h * a.nl_sh + qi * a.nl_sq];
        const float y = a.history_lse[b * a.hl_sb + h * a.hl_sh + qi * a.hl_sq];
        const float m = fmaxf(x, y);
        const float wn = expf(x - m), wh = expf(y - m);
        const float nv =
            bf16_bits_to_f32(a.native[b * a.n_sb + h * a.n_sh + qi * a.n_sq + o * a.n_sd]);
        a.out[(((int64_t)b * a.H + h) * a.Q + qi) * 128 + o] =
            f32_to_bf16_bits((nv * wn + acc * wh) / (wn + wh));
    }
}

// The same on bf16 MFMA, for rows of unit stride in 16-byte pieces.  A wave
// owns 32 queries of one (b, h); the lift is the MFMA's row operand, staged
// transposed in LDS once per 128 queries, the low rows its columns, so a lane
// ends with one query and reads and writes 16 consecutive outputs (32 bytes) of
// each 32-wide tile.
//   Main:  rows of tile n in the order o = 32n + 16 ((p >> 2) & 1) + 4 (p >> 3) +
//          (p & 3) of MFMA row p, which makes a lane's 16 rows consecutive.
//   PRoPE: one product per coordinate c over the quartets (zero-padded to 16),
//          rows j; output 4 j + c.  (Not one product with a block matrix: its
//          zeros would turn an infinity of one coordinate into NaN in all.)
// Products of bf16 are exact in fp32 and summed in fp32, as above.  Bound by
// memory: 2 x 16 x 1,560 rows of low_dim 64 (33 MB) took 72 us with one thread
// per output reading both factors of each product from LDS, now 12 us.
constexpr int LM_WAVES = 4;

template <int K>
__global__ void __launch_bounds__(64 * LM_WAVES) lift_mfma_kernel(nkv_lift_combine_args a) {
    constexpr int KQ = K / 4, QS = (KQ + 15) / 16, LD = K + 8, LDQ = 16 * QS + 8;
    __shared__ __align__(16) uint16_t w[128 * LD > 32 * LDQ ? 128 * LD : 32 * LDQ];
    const int t = threadIdx.x, lane = t & 63, hf = lane >> 5, l32 = lane & 31;
    const int b = (int)(blockIdx.y / a.H), h = (int)(blockIdx.y % a.H);
    const bool prope = b >= a.B;
    const int64_t q0 = (int64_t)blockIdx.x * (32 * LM_WAVES) + 32 * (t >> 6);
    const int64_t qi = min(q0 + l32, a.Q - 1);
    // this lane's loads first: its query's low row, native row and LSEs
    const uint16_t* lp = a.low + b * a.l_sb + h * a.l_sh + qi * a.l_sq;
    const uint16_t* np = a.native + b * a.n_sb + h * a.n_sh + qi * a.n_sq + 16 * hf;
    // the low row's 16-byte pieces: Main, piece hf of each 16; PRoPE, the 32
    // values (8 quartets) hf of each 64
    constexpr int LP = K / 16 > 4 * QS ? K / 16 : 4 * QS;
    u32x4 lr[LP], nr[4][2];
#pragma unroll
    for (int i = 0; i < LP; ++i) {
        const int at = prope ? 64 * (i / 4) + 32 * hf + 8 * (i % 4) : 16 * i + 8 * hf;
        lr[i] = u32x4{0, 0, 0, 0};
        if (at < K) lr[i] = *reinterpret_cast<const u32x4*>(lp + at);
    }
#pragma unroll
    for (int n = 0; n < 4; ++n)
#pragma unroll
        for (int e = 0; e < 2; ++e) nr[n][e] = *reinterpret_cast<const u32x4*>(np + 32 * n + 8 * e);
    const float x = a.native_lse[b * a.nl_sb + h * a.nl_sh + qi * a.nl_sq];
    const float y = a.history_lse[b * a.hl_sb + h * a.hl_sh + qi * a.hl_sq];
    if (!prope) {
        for (int i = t; i < K * 128; i += 64 * LM_WAVES) {
            const int k = i >> 7, o = i & 127;
            const int p = 8 * ((o >> 2) & 3) + 4 * ((o >> 4) & 1) + (o & 3);
            w[(32 * (o >> 5) + p) * LD + k] = a.main_lift[h * a.ml_sh + k * a.ml_sk + o * a.ml_so];
        }
    } else {
        for (int i = t; i < 16 * QS * 32; i += 64 * LM_WAVES) {
            const int k = i >> 5, j = i & 31;
            w[j * LDQ + k] = k < KQ ? a.prope_mix[h * a.pm_sh + k * a.pm_sk + j * a.pm_so] : 0;
        }
    }
    __syncthreads();
    f32x16 acc[4] = {};
    if (!prope) {
#pragma unroll
        for (int s = 0; s < K / 16; ++s)
#pragma unroll
            for (int n = 0; n < 4; ++n)
                acc[n] = mfma32(lds_b128(w + (32 * n + l32) * LD + 16 * s + 8 * hf), as_bf16x8(lr[s]), acc[n]);
    } else {
#pragma unroll
        for (int s = 0; s < QS; ++s) {
            const bf16x8 mix = lds_b128(w + l32 * LDQ + 16 * s + 8 * hf);
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                u32x4 f;   // coordinate c of quartets 0 .. 8
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t q0w = lr[4 * s + i][c >> 1], q1w = lr[4 * s + i][2 + (c >> 1)];
                    f[i] = (c & 1) ? (q0w >> 16) | (q1w & 0xffff0000u) : (q0w & 0xffffu) | (q1w << 16);
                }
                acc[c] = mfma32(mix, as_bf16x8(f), acc[c]);
            }
        }
    }
    if (q0 + l32 >= a.Q) return;
    const float m = fmaxf(x, y);
    const float wn = expf(x - m), wh = expf(y - m), den = wn + wh;
    uint16_t* op = a.out + (((int64_t)b * a.H + h) * a.Q + qi) * 128 + 16 * hf;
#pragma unroll
    for (int n = 0; n < 4; ++n)
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            u32x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float r[2];
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const int i = 8 * g + 2 * e + u;   // of the tile's 16
                    const float lifted = prope ? acc[i & 3][4 * n + (i >> 2)] : acc[n][i];
                    const uint32_t nw = nr[n][g][e];
                    const float nv = __uint_as_float(u ? nw & 0xffff0000u : nw << 16);
                    r[u] = (nv * wn + lifted * wh) / den;
                }
                o[e] = pack_bf16x2(r[0], r[1]);
            }
            *reinterpret_cast<u32x4*>(op + 32 * n + 8 * g) = o;
        }
}

// ---- nkv_finish (LBF:10-34)
// One wave per (b, group head g, s) row; lanes stride over d.  Each lane
// reads its elements' native values before it writes them, so result may
// alias native.
constexpr int FN_WAVES = 4;

__global__ void __launch_bounds__(64 * FN_WAVES) finish_kernel(nkv_finish_args a) {
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * FN_WAVES + (threadIdx.x >> 6);
    const int64_t rows = (int64_t)a.B * a.H_group * a.S;
    if (row >= rows) return;
    const int64_t s = row % a.S;
    const int g = (int)((row / a.S) % a.H_group);
    const int b = (int)(row / ((int64_t)a.S * a.H_group));
    const int hd = a.heads[g];
    // a head index outside the native heads (a corrupt map) writes nothing
    if (hd < 0 || hd >= a.H_native) return;
    const float x = a.native_lse[b * a.la_sb + hd * a.la_sh + s * a.la_ss];
    const float z = a.low_lse[b * a.lb_sb + g * a.lb_sh + s * a.lb_ss];
    float l = fmaxf(x, z) + log1pf(expf(-fabsf(x - z)));
    if (x == z && fabsf(x) == INFINITY) l = x;
    const float origin = fabsf(l) != INFINITY ? l : 0.0f;
    const float ea = expf(x - origin), eb = expf(z - origin);
    const bool correct = a.mean != nullptr;
    const uint16_t* arow = a.native + b * a.a_sb + hd * a.a_sh + s * a.a_ss;
    const uint16_t* brow = a.lifted + b * a.b_sb + g * a.b_sh + s * a.b_ss;
    uint16_t* yrow = a.result + b * a.y_sb + hd * a.y_sh + s * a.y_ss;
    for (int d = lane; d < a.D; d += 64) {
        const float av = bf16_bits_to_f32(arow[d * a.a_sd]);
        float bv = bf16_bits_to_f32(brow[d * a.b_sd]);
        if (correct)
            bv = (bv + a.mean[b * a.m_sb + hd * a.m_sh + d * a.m_sd]) -
                 a.projected[b * a.p_sb + g * a.p_sh + d * a.p_sd];
        yrow[d * a.y_sd] = f32_to_bf16_bits(av * ea + bv * eb);
    }
}

}  // namespace

}  // namespace nkv

using namespace nkv;

extern "C" int nkv_lift_lse_combine(void* stream, const nkv_lift_combine_args* a) {
    NKV_REQUIRE(a, NKV_ERR_INVALID, "null arguments");
    NKV_REQUIRE(a->B >= 0 && a->H >= 1 && a->Q >= 0, NKV_ERR_INVALID, "bad shape");
    NKV_REQUIRE(a->low_dim == 32 || a->low_dim == 64 || a->low_dim == 96, NKV_ERR_UNSUPPORTED,
                "the fused lift supports low_dim 32, 64 and 96");
    if (a->B == 0 || a->Q == 0) return NKV_OK;
    NKV_REQUIRE(a->native && a->native_lse && a->low && a->main_lift && a->prope_mix &&
                    a->history_lse && a->out,
                NKV_ERR_INVALID, "null pointer");
    const int64_t heads = 2 * (int64_t)a->B * a->H;
    NKV_REQUIRE(heads <= 65535, NKV_ERR_UNSUPPORTED, "at most 65535 batch x head pairs");
    // MFMA for rows of unit stride in 16-byte pieces; any other stride one
    // element at a time, as are up to four queries of low_dim 32, whose few
    // products take less than staging the lift transposed (24 heads, us in a
    // graph: 1 query 4.9, by MFMA 6.4; 4 queries 5.75, 6.4; 8 queries 7.2, 6.3;
    // low_dim 64, 1 query 7.3, 7.0)
    if ((a->low_dim > 32 || a->Q > 4) && a->n_sd == 1 && a->l_sd == 1 && rows16(a->native, a->n_sb, a->n_sh, a->n_sq) &&
        rows16(a->low, a->l_sb, a->l_sh, a->l_sq) && reinterpret_cast<uintptr_t>(a->out) % 16 == 0) {
        const dim3 grid((unsigned)cdiv(a->Q, 32 * LM_WAVES), (unsigned)heads);
        auto run = [&](auto kernel) { kernel<<<grid, 64 * LM_WAVES, 0, (hipStream_t)stream>>>(*a); };
        if (a->low_dim == 32) run(lift_mfma_kernel<32>);
        else if (a->low_dim == 64) run(lift_mfma_kernel<64>);
        else run(lift_mfma_kernel<96>);
        NKV_LAUNCH_CHECK();
        return NKV_OK;
    }
    lift_combine_kernel<<<dim3((unsigned)cdiv(a->Q, LC_Q), (unsigned)heads), LC_THREADS, 0,
                          (hipStream_t)stream>>>(*a);
    NKV_LAUNCH_CHECK();
    return NKV_OK;
}

extern "C" int nkv_finish(void* stream, const nkv_finish_args* a) {
    NKV_REQUIRE(a, NKV_ERR_INVALID, "null arguments");
    NKV_REQUIRE(a->B >= 0 && a->H_native >= 1 && a->H_group >= 0 && a->S >= 0 && a->D >= 1,
                NKV_ERR_INVALID, "bad shape");
    NKV_REQUIRE((a->mean == nullptr) == (a->projected == nullptr), NKV_ERR_INVALID,
                "mean and projected come together (the value-mean correction) or not at all");
    const int64_t rows = (int64_t)a->B * a->H_group * a->S;
    if (rows == 0) return NKV_OK;
    NKV_REQUIRE(a->native && a->native_lse && a->lifted && a->low_lse && a->heads && a->result,
                NKV_ERR_INVALID, "null pointer");
    finish_kernel<<<dim3((unsigned)cdiv(rows, FN_WAVES)), 64 * FN_WAVES, 0, (hipStream_t)stream>>>(
        *a);
    NKV_LAUNCH_CHECK();
    return NKV_OK;
}
