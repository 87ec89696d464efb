// nkv_codec.hip -- NanoKV chunk codec on gfx950: INT4 quantise/pack, unpack,
// nearest-center assignment, encoder projection and full-width decode.
//
// This translation unit is compiled with -ffp-contract=off: the quantiser and
// the decode epilogue are bit-exact restatements whose rounding points must
// not be fused away.
#include "nkv_common.h"

#include <type_traits>

namespace nkv {

// ============================================================ quantiser
// quant_lanes(group) lanes of a wave share one (row, group): each takes runs
// of 8 coefficients (two 16-byte loads, whole rows coalesced over the wave),
// the exact amax (order-free) meets by lane exchanges, and every run becomes
// one dword of codes; lane 0 of the group stores the IEEE-divided scale.  (One
// thread per group read a row stride per load and had 1,560 threads for a
// chunk with one scale per row: 51 us at r = 384, now 4.)  Reference:
// MG:349-351 (fp32 arithmetic as in HY kv_codecs.py:244-255; bf16 arithmetic
// as MG deploys it) and _pack_int4 MG:282-292.
__host__ __device__ __forceinline__ int quant_lanes(int group) {
    int n = 1;
    while (n < 64 && 8 * n < group) n *= 2;
    return n;
}

// Lane `sub` of the lpg lanes (aligned in the wave) of group gid; every lane
// of the wave calls.
template <int QUANT_MODE>
__device__ __forceinline__ void quant_pack_group(const float* __restrict__ coeff, int64_t rows,
                                                 int r, int group, int scale_dtype,
                                                 uint8_t* __restrict__ packed,
                                                 uint16_t* __restrict__ scales, int64_t gid,
                                                 int sub, int lpg) {
    const int ngroups = r / group;
    const bool ok = gid < rows * ngroups;
    const int64_t row = ok ? gid / ngroups : 0;
    const int g = ok ? (int)(gid - row * ngroups) : 0;
    const float* x = coeff + row * r + (int64_t)g * group;

    float amax = 0.0f;
    f32x4 v0 = {}, v1 = {};
    for (int j = 8 * sub; ok && j < group; j += 8 * lpg) {
        v0 = *reinterpret_cast<const f32x4*>(x + j);
        v1 = *reinterpret_cast<const f32x4*>(x + j + 4);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float v = e < 4 ? v0[e] : v1[e - 4];
            float a = QUANT_MODE == NKV_QUANT_BF16 ? bf16_round(v) : v;
            a = fabsf(a);
            amax = (a > amax || a != a) ? a : amax;  // NaN propagates like torch.amax
        }
    }
    for (int off = 1; off < lpg; off <<= 1) {
        const float o = __shfl_xor(amax, off);
        amax = (o > amax || o != o) ? o : amax;
    }
    if (!ok) return;
    float s;
    const float eps = 1.1920928955078125e-07f;  // torch.finfo(torch.float32).eps
    float clamped = (amax > eps || amax != amax) ? amax : eps;
    if (QUANT_MODE == NKV_QUANT_BF16) {
        s = bf16_round(__fdiv_rn(bf16_round(clamped), 7.0f));
    } else {
        s = __fdiv_rn(clamped, 7.0f);
    }
    if (sub == 0)
        scales[row * ngroups + g] =
            scale_dtype == NKV_DTYPE_FP16 ? f32_to_f16_bits(s) : f32_to_bf16_bits(s);

    uint8_t* out = packed + row * (r / 2) + (int64_t)g * (group / 2);
    for (int j = 8 * sub; j < group; j += 8 * lpg) {
        if (group > 8 * lpg) {  // more than one run per lane: read again
            v0 = *reinterpret_cast<const f32x4*>(x + j);
            v1 = *reinterpret_cast<const f32x4*>(x + j + 4);
        }
        uint32_t word = 0;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            float v = e < 4 ? v0[e] : v1[e - 4];
            if (QUANT_MODE == NKV_QUANT_BF16) v = bf16_round(v);
            float q = __fdiv_rn(v, s);
            if (QUANT_MODE == NKV_QUANT_BF16) q = bf16_round(q);
            float rq = rintf(q);  // round half to even, as torch.round
            int c = rq != rq ? 0 : (int)fminf(fmaxf(rq, -7.0f), 7.0f);
            word |= (uint32_t)(c + 7) << (4 * e);
        }
        *reinterpret_cast<uint32_t*>(out + j / 2) = word;
    }
}

template <int QUANT_MODE>
__global__ void __launch_bounds__(256) quant_pack_kernel(const float* __restrict__ coeff,
                                                         int64_t rows, int r, int group,
                                                         int scale_dtype,
                                                         uint8_t* __restrict__ packed,
                                                         uint16_t* __restrict__ scales) {
    const int lpg = quant_lanes(group), t = threadIdx.x;
    quant_pack_group<QUANT_MODE>(coeff, rows, r, group, scale_dtype, packed, scales,
                                 (int64_t)blockIdx.x * (256 / lpg) + t / lpg, t % lpg, lpg);
}

// ============================================================ unpack
// One thread per 8 consecutive codes (4 packed bytes) of one row.
__global__ void __launch_bounds__(256) unpack_kernel(const uint8_t* __restrict__ packed,
                                                     const uint16_t* __restrict__ scales,
                                                     int scale_dtype,
                                                     const int32_t* __restrict__ row_index,
                                                     int64_t rows, int r, int group,
                                                     uint16_t* __restrict__ out) {
    const int per_row = r / 8;
    const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (tid >= rows * per_row) return;
    const int64_t i = tid / per_row;
    const int j0 = (int)(tid - i * per_row) * 8;
    const int64_t src = row_index ? (int64_t)row_index[i] : i;
    const uint32_t word = *reinterpret_cast<const uint32_t*>(packed + src * (r / 2) + j0 / 2);
    const float s = scale_bits_to_f32(scales[src * (r / group) + j0 / group], scale_dtype);
    u32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float lo = (float)((int)((word >> (8 * e)) & 15u) - 7) * s;
        float hi = (float)((int)((word >> (8 * e + 4)) & 15u) - 7) * s;
        o[e] = pack_bf16x2(lo, hi);
    }
    *reinterpret_cast<u32x4*>(out + i * r + j0) = o;
}

// ============================================================ assignment
// fp64 nearest-center search.  A 256-thread block owns 32 rows and walks the
// center table in chunks of 64; each thread keeps a 2-row x 4-center fp64
// register tile.  Per chunk the block stages x[32 x 64] (fp32) and
// c[64 x 64] (bf16) in LDS along HD.  ||c||^2 is accumulated by the same
// threads (only the thread column that owns row 0 keeps it).  Distances are
// ||c||^2 - 2 x.c (||x||^2 is constant per row); ties keep the lowest index.
constexpr int AS_ROWS = 32, AS_CENT = 64, AS_K = 64;

template <int ID_BYTES>
__device__ __forceinline__ void store_id(void* ids, int64_t i, int v) {
    if (ID_BYTES == 1) reinterpret_cast<uint8_t*>(ids)[i] = (uint8_t)v;
    else if (ID_BYTES == 2) reinterpret_cast<uint16_t*>(ids)[i] = (uint16_t)v;
    else reinterpret_cast<int32_t*>(ids)[i] = v;
}

// A center element as fp32: bf16 bits or fp32 (both exact in fp64).
__device__ __forceinline__ float center_value(const uint16_t* c, int64_t i) {
    return bf16_bits_to_f32(c[i]);
}
__device__ __forceinline__ float center_value(const float* c, int64_t i) { return c[i]; }

template <int ID_BYTES, typename CT = uint16_t>
__global__ void __launch_bounds__(256) assign_kernel(const float* __restrict__ x,
                                                     const CT* __restrict__ centers,
                                                     int64_t rows, int C, int HD,
                                                     void* __restrict__ ids) {
    __shared__ float xs[AS_ROWS][AS_K + 1];
    __shared__ float cs[AS_CENT][AS_K + 1];
    __shared__ double red_d[AS_ROWS][16];
    __shared__ int red_c[AS_ROWS][16];

    const int t = threadIdx.x;
    const int tr = t / 16;          // rows tr and tr + 16
    const int tc = t % 16;          // centers tc + 16*j, j = 0..3
    const int64_t row0 = (int64_t)blockIdx.x * AS_ROWS;

    double best[2] = {0.0, 0.0};
    int best_c[2] = {-1, -1};

    for (int c0 = 0; c0 < C; c0 += AS_CENT) {
        double dot[2][4] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
        double cc[4] = {0, 0, 0, 0};
        for (int k0 = 0; k0 < HD; k0 += AS_K) {
            __syncthreads();
            // stage x: 32 x 64 fp32 = 2048 values, 8 per thread
            for (int e = t; e < AS_ROWS * AS_K; e += 256) {
                int rr = e / AS_K, kk = e % AS_K;
                int64_t gr = row0 + rr;
                xs[rr][kk] = (gr < rows && k0 + kk < HD) ? x[gr * HD + k0 + kk] : 0.0f;
            }
            for (int e = t; e < AS_CENT * AS_K; e += 256) {
                int cr = e / AS_K, kk = e % AS_K;
                int gc = c0 + cr;
                cs[cr][kk] = (gc < C && k0 + kk < HD)
                                 ? center_value(centers, (int64_t)gc * HD + k0 + kk)
                                 : 0.0f;
            }
            __syncthreads();
            for (int kk = 0; kk < AS_K; ++kk) {
                double xv0 = (double)xs[tr][kk];
                double xv1 = (double)xs[tr + 16][kk];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    double cv = (double)cs[tc + 16 * j][kk];
                    dot[0][j] += xv0 * cv;
                    dot[1][j] += xv1 * cv;
                    cc[j] += cv * cv;
                }
            }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            int c = c0 + tc + 16 * j;
            if (c >= C) continue;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                double d = cc[j] - 2.0 * dot[i][j];
                if (best_c[i] < 0 || d < best[i] || (d == best[i] && c < best_c[i])) {
                    best[i] = d;
                    best_c[i] = c;
                }
            }
        }
    }
    // reduce over the 16 center lanes of each row (fixed order: lowest index wins ties)
    red_d[tr][tc] = best[0];
    red_c[tr][tc] = best_c[0];
    red_d[tr + 16][tc] = best[1];
    red_c[tr + 16][tc] = best_c[1];
    __syncthreads();
    if (t < AS_ROWS) {
        double bd = red_d[t][0];
        int bc = red_c[t][0];
        for (int j = 1; j < 16; ++j) {
            int c = red_c[t][j];
            double d = red_d[t][j];
            if (c >= 0 && (bc < 0 || d < bd || (d == bd && c < bc))) {
                bd = d;
                bc = c;
            }
        }
        int64_t gr = row0 + t;
        if (gr < rows) store_id<ID_BYTES>(ids, gr, bc);
    }
}

// fp64 MFMA nearest-center search (v_mfma_f64_16x16x4_f64).  A 256-thread
// block owns 16 rows; wave w takes centers 64*w + [0, 64) of every group of
// 256 as four 16 x 16 output tiles.  Operands come straight from L2: at each
// 16-wide k block lane l supplies x row (l % 16) and center column (l % 16)
// at k = k0 + 4*(l / 16) + [0, 4), one 16-byte x piece and one 8-byte
// center piece per tile for four MFMA steps (any k order is valid for the
// reduction, and A and B use the same one).  Every product of an fp32 x and
// a bf16 center is exact in fp64, so only the order of the fp64 sums differs
// from the fp64 VALU search (relative 1e-16).  ||c||^2 comes from the same
// center pieces.  Output layout: lane l, element e holds row 4e + l/16,
// column l % 16.  Needs HD % 16 == 0, x 16-byte and centers 8-byte aligned.
constexpr int AM_ROWS = 16, AM_AHEAD = 4;
typedef double f64x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ bool better(double d, int c, double bd, int bc) {
    return bc < 0 || (c >= 0 && (d < bd || (d == bd && c < bc)));
}

// Four consecutive center elements of one lane's k block: 8 bytes of bf16
// or 16 bytes of fp32; element st as an exact fp64.
template <typename CT>
struct CenterPiece;
template <>
struct CenterPiece<uint16_t> {
    using V = u32x2;
    static __device__ __forceinline__ double get(const V& v, int st) {
        const uint32_t w = v[st >> 1];
        return (double)__uint_as_float((st & 1) ? (w & 0xffff0000u) : (w << 16));
    }
};
template <>
struct CenterPiece<float> {
    using V = u32x4;
    static __device__ __forceinline__ double get(const V& v, int st) {
        return (double)__uint_as_float(v[st]);
    }
};

template <int ID_BYTES, typename CT = uint16_t>
__global__ void __launch_bounds__(256) assign_mfma_kernel(const float* __restrict__ x,
                                                          const CT* __restrict__ centers,
                                                          int64_t rows, int C, int HD,
                                                          void* __restrict__ ids) {
    using CP = CenterPiece<CT>;
    __shared__ double red_d[4][AM_ROWS];
    __shared__ int red_c[4][AM_ROWS];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int g = lane >> 4, col = lane & 15;
    const int64_t row0 = (int64_t)blockIdx.x * AM_ROWS;
    const int64_t xr = min(row0 + col, rows - 1);  // rows past the end read the last row
    const float* xp = x + xr * HD + 4 * g;
    double bd[4];
    int bc[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) { bd[e] = 0.0; bc[e] = -1; }

    for (int cg = 0; cg < C; cg += 256) {
        const CT* cp[4];
        int cid[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            cid[t] = cg + 64 * wave + 16 * t + col;
            cp[t] = centers + (int64_t)min(cid[t], C - 1) * HD + 4 * g;
        }
        f64x4 acc[4];
        double cc[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) { acc[t] = f64x4{0.0, 0.0, 0.0, 0.0}; cc[t] = 0.0; }
        // a ring of AM_AHEAD k blocks of operands in flight (one k block =
        // 16 k: four MFMA steps per tile); block kb lives in slot kb % AM_AHEAD
        const int NB = HD / 16;
        u32x4 xa[AM_AHEAD];
        typename CP::V cb[AM_AHEAD][4];
        auto issue = [&](int kb, int slot) {
            xa[slot] = *reinterpret_cast<const u32x4*>(xp + 16 * kb);
#pragma unroll
            for (int t = 0; t < 4; ++t)
                cb[slot][t] = *reinterpret_cast<const typename CP::V*>(cp[t] + 16 * kb);
        };
#pragma unroll
        for (int i = 0; i < AM_AHEAD; ++i)
            if (i < NB) issue(i, i);
        for (int kb0 = 0; kb0 < NB; kb0 += AM_AHEAD) {
#pragma unroll
            for (int i = 0; i < AM_AHEAD; ++i) {
                const int kb = kb0 + i;
                if (kb >= NB) break;
                const u32x4 xv = xa[i];
                typename CP::V cv[4];
#pragma unroll
                for (int t = 0; t < 4; ++t) cv[t] = cb[i][t];
                if (kb + AM_AHEAD < NB) issue(kb + AM_AHEAD, i);
#pragma unroll
                for (int st = 0; st < 4; ++st) {
                    const double a = (double)__uint_as_float(xv[st]);
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        const double b = CP::get(cv[t], st);
                        acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc[t], 0, 0, 0);
                        cc[t] = fma(b, b, cc[t]);
                    }
                }
            }
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            // ||c||^2 over the four k subsets of this column
            cc[t] += __shfl_xor(cc[t], 16);
            cc[t] += __shfl_xor(cc[t], 32);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const double d = cc[t] - 2.0 * acc[t][e];
                const int c = cid[t] < C ? cid[t] : -1;
                if (better(d, c, bd[e], bc[e])) { bd[e] = d; bc[e] = c; }
            }
        }
    }
    // lanes of one row group (same g) hold rows 4e + g: reduce over columns
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int off = 1; off < 16; off <<= 1) {
            const double od = __shfl_xor(bd[e], off);
            const int oc = __shfl_xor(bc[e], off);
            if (better(od, oc, bd[e], bc[e])) { bd[e] = od; bc[e] = oc; }
        }
    if (col == 0) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            red_d[wave][4 * e + g] = bd[e];
            red_c[wave][4 * e + g] = bc[e];
        }
    }
    __syncthreads();
    if (threadIdx.x < AM_ROWS) {
        const int r = threadIdx.x;
        double d = red_d[0][r];
        int c = red_c[0][r];
        for (int w = 1; w < 4; ++w)
            if (better(red_d[w][r], red_c[w][r], d, c)) { d = red_d[w][r]; c = red_c[w][r]; }
        const int64_t gr = row0 + r;
        if (gr < rows) store_id<ID_BYTES>(ids, gr, c);
    }
}

// bf16 MFMA nearest-center search with an exact decision (C <= 256).
// x = hi + lo + r with hi = bf16(x), lo = bf16(x - hi), |r| <= 2^-16 |x|;
// the centers are exact bf16, so the two MFMA passes hi.c and lo.c have
// exact products and only fp32 sums.  The MFMA accumulator restarts every
// AB_SEG k values and the segment sums are added in a second fp32
// accumulator, so even with one fp32 rounding per addition the dot product
// is within (g_2SEG + g_nseg)(1 + 2^-7) + 2^-16 < 5e-5 of sum |x||c| <=
// ||x|| ||c|| (g_n = n 2^-24 / (1 - n 2^-24), nseg = HD / SEG <= 64);
// ||c||^2 is summed the same way (fp32 per segment, fp64 across: < 1e-5
// ||c||^2).  With the final fp32 subtraction every approximate distance
// dt_c = ||c||^2 - 2 x.c is within 1.1e-4 (||x|| ||c|| + ||c||^2) of the
// exact one (2e-4 if the matrix core truncated instead of rounding); the
// search uses
//   E_c = AB_KAPPA (||x|| ||c|| + ||c||^2),   AB_KAPPA = 2.5e-4,
// With U = min_c (dt_c + E_c) the exact argmin is among the candidates
// {c : dt_c - E_c <= U}; a row with one candidate is decided, a row with
// several re-evaluates just those in fp64 (exact products, first index on
// ties), the arithmetic of assign_kernel.
// A 512-thread block owns 32 rows; wave w takes centers 32w + [0, 32) as one
// 32 x 32 tile.  x is split into hi/lo bf16 tiles in LDS per 128-wide k
// chunk (shared by the eight waves); center fragments come from L2 one chunk
// ahead.  Needs HD % AB_SEG == 0, HD <= AB_MAXK, C <= 256, x and centers
// 16-byte aligned.
constexpr int AB_ROWS = 32, AB_KC = 128, AB_SEG = 256, AB_MAXC = 256, AB_WAVES = 8, AB_MAXK = 16384;
constexpr float AB_KAPPA = 2.5e-4f;

// ------------------------------------------------ batched encode problems
// One launch per encode stage serves up to ENC_MAXB independent problems of
// one shape (K and V of a layer, batch items): problem blockIdx.y (search,
// quantiser) or blockIdx.z (projection).  A problem's rows are fp32 (x) or
// bf16 (xb, read as the reference's value.float(): exact), row stride ldx.
constexpr int ENC_MAXB = 8;
struct EncProb {
    const float* x;
    const uint16_t* xb;
    int64_t ldx;
    const uint16_t* centers;
    void* ids;
    const float* mean;
    const uint16_t* w_enc;
    float* coeff;
    uint8_t* packed;
    uint16_t* scales;
    int64_t M;
};
struct EncBatch {
    EncProb p[ENC_MAXB];
    int n, K, r, num_centers, id_bytes;
    int64_t row_blocks;   // 32-row blocks of the largest problem (set per launch)
    // the quantiser run inside the projection: group size (0: separate
    // launch), scale dtype and NKV_QUANT_* mode
    int qgroup, scale_dtype, quant_mode;
    // center id of row m of problem p (clamped into the table)
    __device__ __forceinline__ int id_of(const EncProb& q, int64_t m) const {
        int v;
        if (id_bytes == 1) v = reinterpret_cast<const uint8_t*>(q.ids)[m];
        else if (id_bytes == 2) v = reinterpret_cast<const uint16_t*>(q.ids)[m];
        else v = reinterpret_cast<const int32_t*>(q.ids)[m];
        return min(max(v, 0), num_centers - 1);
    }
};

// Eight consecutive input values of one row (16-byte loads), held raw until
// they are used.
template <bool XB>
struct X8 {
    u32x4 w[XB ? 1 : 2];
    __device__ __forceinline__ void load(const EncProb& q, int64_t m, int k) {
        if constexpr (XB) {
            w[0] = *reinterpret_cast<const u32x4*>(q.xb + m * q.ldx + k);
        } else {
            const float* r = q.x + m * q.ldx + k;
            w[0] = *reinterpret_cast<const u32x4*>(r);
            w[1] = *reinterpret_cast<const u32x4*>(r + 4);
        }
    }
    __device__ __forceinline__ float operator[](int e) const {
        if constexpr (XB)
            return __uint_as_float((e & 1) ? (w[0][e >> 1] & 0xffff0000u) : (w[0][e >> 1] << 16));
        else
            return __uint_as_float(w[e >> 2][e & 3]);
    }
};

// Work item of block blk when a launch's items are cut into eight equal runs,
// one per XCD (blocks are dispatched to the XCDs round-robin): block blk runs
// slot blk / 8 of XCD blk % 8.  Items that share operands (one problem's
// centers, one W_enc column slice) are numbered together, so they meet in
// one XCD's L2.  Blocks past the last item get an item >= items.
__device__ __forceinline__ int64_t xcd_item(int64_t blk, int64_t items) {
    const int64_t per = (items + 7) >> 3;
    return (blk & 7) * per + (blk >> 3);
}
static inline unsigned xcd_grid(int64_t items) { return (unsigned)(8 * ((items + 7) >> 3)); }

// The quantiser over every problem of a batch (problem blockIdx.y).
template <int QUANT_MODE>
__global__ void __launch_bounds__(256) quant_pack_batch_kernel(EncBatch B, int group,
                                                               int scale_dtype) {
    const EncProb& P = B.p[blockIdx.y];
    const int lpg = quant_lanes(group), t = threadIdx.x;
    quant_pack_group<QUANT_MODE>(P.coeff, P.M, B.r, group, scale_dtype, P.packed, P.scales,
                                 (int64_t)blockIdx.x * (256 / lpg) + t / lpg, t % lpg, lpg);
}

// The search's small block state: ||x||^2 per row, the per-wave bounds U,
// and each row's candidate count, first candidate and candidate bit set.
struct AssignSmall {
    float xn[AB_ROWS];
    float red[AB_WAVES][AB_ROWS];
    int cnt[AB_ROWS], first[AB_ROWS];
    uint32_t cand[AB_ROWS][AB_MAXC / 32];
};

__device__ __forceinline__ void assign_small_init(AssignSmall& sm, int t) {
    if (t < AB_ROWS) { sm.xn[t] = 0.0f; sm.cnt[t] = 0; sm.first[t] = 0x7fffffff; }
    for (int e = t; e < AB_ROWS * AB_MAXC / 32; e += 64 * AB_WAVES) (&sm.cand[0][0])[e] = 0u;
}

// ||c||^2 - 2 x.c of row gr in fp64 (exact products), by the whole wave: 8
// consecutive values per lane and step, four steps' loads issued together,
// summed in ascending k per lane, then over the lanes.
template <bool XB>
__device__ __forceinline__ double exact_distance(const EncProb& P, const uint16_t* cr, int64_t gr,
                                                 int HD, int lane) {
    double cc = 0.0, xc = 0.0;
    for (int k = 8 * lane; k < HD; k += 4 * 512) {
        u32x4 cw[4];
        X8<XB> x8[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (k + 512 * u < HD) {
                cw[u] = *reinterpret_cast<const u32x4*>(cr + k + 512 * u);
                x8[u].load(P, gr, k + 512 * u);
            }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (k + 512 * u >= HD) break;
            const uint32_t w4[4] = {cw[u].x, cw[u].y, cw[u].z, cw[u].w};
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const uint32_t hb = (e & 1) ? (w4[e >> 1] & 0xffff0000u) : (w4[e >> 1] << 16);
                const double cv = (double)__uint_as_float(hb);
                cc = fma(cv, cv, cc);
                xc = fma((double)x8[u][e], cv, xc);
            }
        }
    }
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        cc += __shfl_xor(cc, off);
        xc += __shfl_xor(xc, off);
    }
    return cc - 2.0 * xc;
}

// The decision after the products: tot (this lane's 16 dot products x.c,
// rows 8(i/4) + 4hf + i%4 of the block, center col), cnf = ||c||^2, and
// sm.xn complete.  Rows with one candidate are decided; the others compare
// their candidates exactly in fp64 (one wave per row, lanes split HD).
template <int ID_BYTES, bool XB>
__device__ __forceinline__ void assign_finish(const EncBatch& B, const EncProb& P, AssignSmall& sm,
                                              const f32x16& tot, float cnf, int col, int64_t row0) {
    const int64_t rows = P.M;
    const int C = B.num_centers, HD = B.K;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int hf = lane >> 5, l32 = lane & 31;
    float dt[16], ee[16];
    {
        const float cnorm = sqrtf(cnf) * 1.001f;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int r = 8 * (i / 4) + 4 * hf + (i % 4);
            const float xnorm = sqrtf(sm.xn[r]) * 1.001f;
            dt[i] = col < C ? cnf - 2.0f * tot[i] : INFINITY;
            ee[i] = AB_KAPPA * (xnorm * cnorm + cnf * 1.001f);
        }
    }
    // U = min over the row's columns of dt + E: a half-wave holds a row's 32 columns
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        float u = dt[i] + ee[i];
#pragma unroll
        for (int off = 1; off < 32; off <<= 1) u = fminf(u, __shfl_xor(u, off));
        if (l32 == 0) sm.red[wave][8 * (i / 4) + 4 * hf + (i % 4)] = u;
    }
    __syncthreads();
    // candidates: those not above U
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int r = 8 * (i / 4) + 4 * hf + (i % 4);
        float U = sm.red[0][r];
#pragma unroll
        for (int w = 1; w < AB_WAVES; ++w) U = fminf(U, sm.red[w][r]);
        if (col < C && !(dt[i] - ee[i] > U)) {
            atomicAdd(&sm.cnt[r], 1);
            atomicMin(&sm.first[r], col);
            atomicOr(&sm.cand[r][col >> 5], 1u << (col & 31));
        }
    }
    __syncthreads();
    for (int r = wave; r < AB_ROWS; r += AB_WAVES) {
        const int64_t gr = row0 + r;
        if (gr >= rows) continue;
        // Where a sum overflowed (an infinity, or norms past fp32) the bound is
        // NaN and the center stays a candidate, so fp64 decides; a row with a
        // NaN is NaN from every center: 0.
        const bool nan_row = sm.xn[r] != sm.xn[r];
        int best = nan_row ? 0 : sm.first[r];
        if (sm.cnt[r] > 1 && !nan_row) {
            double bd = 0.0;
            best = -1;
            for (int w = 0; w < AB_MAXC / 32; ++w) {
                uint32_t bits = sm.cand[r][w];
                while (bits) {
                    const int c = 32 * w + __builtin_ctz(bits);
                    bits &= bits - 1;
                    const double d = exact_distance<XB>(P, P.centers + (int64_t)c * HD, gr, HD, lane);
                    // (a center with a NaN loses to any other)
                    if (better(d, c, bd, best) || (bd != bd && d == d)) { bd = d; best = c; }
                }
            }
        }
        if (lane == 0) store_id<ID_BYTES>(P.ids, gr, best);
    }
}

template <int ID_BYTES, bool XB>
__global__ void __launch_bounds__(64 * AB_WAVES) assign_bf16_kernel(EncBatch B) {
    const EncProb& P = B.p[blockIdx.y];
    const int64_t rows = P.M;
    const int C = B.num_centers, HD = B.K;
    const uint16_t* __restrict__ centers = P.centers;
    if ((int64_t)blockIdx.x * AB_ROWS >= rows) return;
    __shared__ __align__(16) uint16_t xs[2][AB_ROWS][AB_KC + 8];
    __shared__ AssignSmall sm;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int hf = lane >> 5, l32 = lane & 31;
    const int64_t row0 = (int64_t)blockIdx.x * AB_ROWS;
    assign_small_init(sm, t);
    // fill: thread t splits row t/16, k columns 8*(t%16) .. +8 of each chunk
    const int frow = t >> 4, fk = 8 * (t & 15);
    const int64_t fr = min(row0 + frow, rows - 1);
    const bool frow_ok = row0 + frow < rows;
    // this lane's center column
    const int col = 32 * wave + l32;
    const uint16_t* crow = centers + (int64_t)min(col, C - 1) * HD + 8 * hf;
    f32x16 acc = {}, tot = {};
    float cseg = 0.0f;
    double cn = 0.0;
    float xsq = 0.0f;
    u32x4 bcur[8], bnxt[8];
    X8<XB> xcur, xnxt;
    auto fetch = [&](int kc, u32x4 (&b)[8], X8<XB>& xv) {
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) b[ks] = *reinterpret_cast<const u32x4*>(crow + kc + 16 * ks);
        xv.load(P, fr, kc + fk);
    };
    // one chunk: split x into hi / lo bf16 through LDS, then the MFMAs of
    // both passes and the column norms
    auto body = [&](int kc, const u32x4 (&bq)[8], const X8<XB>& xq) {
        {
            // split this thread's 8 values into hi / lo bf16
            const float v[8] = {xq[0], xq[1], xq[2], xq[3], xq[4], xq[5], xq[6], xq[7]};
            u32x4 hi, lo;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t hp = pack_bf16x2(v[2 * e], v[2 * e + 1]);
                hi[e] = hp;
                lo[e] = pack_bf16x2(v[2 * e] - __uint_as_float(hp << 16),
                                    v[2 * e + 1] - __uint_as_float(hp & 0xffff0000u));
                xsq = fmaf(v[2 * e], v[2 * e], fmaf(v[2 * e + 1], v[2 * e + 1], xsq));
            }
            *reinterpret_cast<u32x4*>(&xs[0][frow][fk]) = hi;
            *reinterpret_cast<u32x4*>(&xs[1][frow][fk]) = lo;
        }
        __syncthreads();
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
            const bf16x8 ah = *reinterpret_cast<const bf16x8*>(&xs[0][l32][16 * ks + 8 * hf]);
            const bf16x8 al = *reinterpret_cast<const bf16x8*>(&xs[1][l32][16 * ks + 8 * hf]);
            const bf16x8 bb = as_bf16x8(bq[ks]);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bb, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al, bb, acc, 0, 0, 0);
            // (the words go through named scalars: indexing the vector inside
            // the bit_cast was lowered to word 0 four times)
            const uint32_t w4[4] = {bq[ks].x, bq[ks].y, bq[ks].z, bq[ks].w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const bf16x2 wv = __builtin_bit_cast(bf16x2, w4[e]);
                cseg = __builtin_amdgcn_fdot2_f32_bf16(wv, wv, cseg, false);
            }
        }
        if ((kc + AB_KC) % AB_SEG == 0) {
            // end of a segment: fold it into the second accumulators
#pragma unroll
            for (int i = 0; i < 16; ++i) tot[i] += acc[i];
            acc = f32x16{};
            cn += (double)cseg;
            cseg = 0.0f;
        }
        __syncthreads();
    };
    // the next chunk's operands (the last chunk reloads itself), issued
    // before this chunk's work and kept there (the fence stops the scheduler
    // from sinking the loads next to their use)
    fetch(0, bcur, xcur);
    __syncthreads();
    for (int kc = 0; kc < HD; kc += AB_KC) {
        fetch(kc + AB_KC < HD ? kc + AB_KC : kc, bnxt, xnxt);
        __builtin_amdgcn_sched_barrier(0);
        body(kc, bcur, xcur);
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) bcur[ks] = bnxt[ks];
        xcur = xnxt;
    }
    // ||x||^2 per row (16 threads per row), ||c||^2 per column (two k halves)
    atomicAdd(&sm.xn[frow], frow_ok ? xsq : 0.0f);
    cn += __shfl_xor(cn, 32);
    const float cnf = (float)cn;
    __syncthreads();
    assign_finish<ID_BYTES, XB>(B, P, sm, tot, cnf, col, row0);
}

// The same search for bf16 rows.  A bf16 x is its own hi part (lo = 0), so
// one MFMA pass gives the products the two-pass form gives, bit for bit.
// Both operands go global -> LDS by 1 KB DMA pieces in 128-wide k stages
// (72 KB: the 256 center rows and the block's 32 input rows, each as
// [row][16 chunks of 16 bytes] with chunk c of row q at slot c ^ (q % 8)),
// double-buffered: after the barrier of stage i the next stage is issued and
// stage i's 8 MFMAs per wave run under it; wave 0 also sums ||x||^2 of its
// fragments.  A block's stream is bound by a fixed cost per barrier plus one
// per 1 KB piece, so few large stages stream faster than many small ones (on
// the box 32 KB stages reached about 100 GB/s per CU, 8 KB stages 38 GB/s,
// whatever the number in flight).  The old form read every center fragment
// straight from L2 (32 rows per load instruction) and waited on it at every
// chunk.
constexpr int AD_KS = 128, AD_NST = 2;
constexpr int AD_CPR = AD_KS / 8;                 // 16-byte chunks per row
constexpr int AD_RPP = 1024 / (AD_KS * 2);        // rows per 1 KB piece
constexpr int AD_CPIECES = AB_MAXC / AD_RPP, AD_PIECES = AD_CPIECES + AB_ROWS / AD_RPP;
constexpr int AD_STAGE = AD_PIECES * 1024;
constexpr int AD_QLO = AD_PIECES / AB_WAVES, AD_NHI = AD_PIECES % AB_WAVES;
constexpr int AD_QMAX = AD_QLO + (AD_NHI ? 1 : 0);
constexpr int AD_SMEM = AD_NST * AD_STAGE;
static_assert(AD_SMEM + (int)sizeof(AssignSmall) <= 160 * 1024, "LDS budget");
static_assert(AB_SEG % AD_KS == 0, "segments are whole stages");
static_assert(AD_NST == 2, "the loop issues one stage ahead");

template <int ID_BYTES>
__global__ void __launch_bounds__(64 * AB_WAVES) assign_dma_kernel(EncBatch B) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ AssignSmall sm;
    // items: (problem, row block), row block fastest
    const int64_t item = xcd_item(blockIdx.x, B.n * B.row_blocks);
    if (item >= B.n * B.row_blocks) return;
    const EncProb& P = B.p[item / B.row_blocks];
    const int64_t rows = P.M;
    const int C = B.num_centers, HD = B.K, S = HD / AD_KS;
    const int64_t row0 = (item % B.row_blocks) * AB_ROWS;
    if (row0 >= rows) return;
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int hf = lane >> 5, l32 = lane & 31;
    assign_small_init(sm, t);
    // this wave's pieces e = wave + AB_WAVES i: center rows AD_RPP e .. (the
    // last row past C), then input rows (the last row past the end); lane L
    // brings slot L % AD_CPR of its row, logical chunk (L % AD_CPR) ^ (row % 8)
    const uint16_t* src[AD_QMAX];
#pragma unroll
    for (int i = 0; i < AD_QMAX; ++i) {
        const int e = wave + AB_WAVES * i;
        const int q = AD_RPP * e + lane / AD_CPR;          // row of the stage image
        const int ch = 8 * ((lane % AD_CPR) ^ (q & 7));
        if (e < AD_CPIECES) {
            src[i] = P.centers + (int64_t)min(q, C - 1) * HD + ch;
        } else {
            const int64_t m = min(row0 + (q - AB_MAXC), rows - 1);
            src[i] = P.xb + m * P.ldx + ch;
        }
    }
    auto issue = [&](int stg) {
        unsigned char* dst = smem_raw + (stg % AD_NST) * AD_STAGE;
#pragma unroll
        for (int i = 0; i < AD_QMAX; ++i)
            if (i < AD_QLO || wave < AD_NHI)
                dma16(src[i] + stg * AD_KS, dst + 1024 * (wave + AB_WAVES * i));
    };
    const int col = 32 * wave + l32;
    f32x16 acc = {}, tot = {};
    float cseg = 0.0f, xsq = 0.0f;
    double cn = 0.0;
    const int xrow_b = (AB_MAXC + l32) * (AD_KS * 2), crow_b = col * (AD_KS * 2);
    issue(0);
    for (int it = 0; it < S; ++it) {
        // stage it landed (nothing later is in flight yet), then the buffer
        // of stage it - 1 is free for stage it + 1
        wait_vmcnt<0>();
        lds_barrier();
        if (it + 1 < S) issue(it + 1);
        const unsigned char* sb = smem_raw + (it % AD_NST) * AD_STAGE;
        bf16x8 af[AD_KS / 16], cf[AD_KS / 16];
#pragma unroll
        for (int k16 = 0; k16 < AD_KS / 16; ++k16) {
            const int slot = 16 * ((2 * k16 + hf) ^ (l32 & 7));
            af[k16] = lds_b128(reinterpret_cast<const uint16_t*>(sb + xrow_b + slot));
            cf[k16] = lds_b128(reinterpret_cast<const uint16_t*>(sb + crow_b + slot));
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k16 = 0; k16 < AD_KS / 16; ++k16) {
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[k16], cf[k16], acc, 0, 0, 0);
            const u32x4 cw = __builtin_bit_cast(u32x4, cf[k16]);
            const uint32_t w4[4] = {cw.x, cw.y, cw.z, cw.w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const bf16x2 wv = __builtin_bit_cast(bf16x2, w4[e]);
                cseg = __builtin_amdgcn_fdot2_f32_bf16(wv, wv, cseg, false);
            }
            if (wave == 0) {
                const u32x4 xw = __builtin_bit_cast(u32x4, af[k16]);
                const uint32_t x4[4] = {xw.x, xw.y, xw.z, xw.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const bf16x2 xv = __builtin_bit_cast(bf16x2, x4[e]);
                    xsq = __builtin_amdgcn_fdot2_f32_bf16(xv, xv, xsq, false);
                }
            }
        }
        if (((it + 1) * AD_KS) % AB_SEG == 0 || it + 1 == S) {
            // end of a segment: fold it into the second accumulators
#pragma unroll
            for (int i = 0; i < 16; ++i) tot[i] += acc[i];
            acc = f32x16{};
            cn += (double)cseg;
            cseg = 0.0f;
        }
    }
    // ||x||^2 per row (wave 0: two k halves), ||c||^2 per column (two k halves)
    if (wave == 0) {
        const float xs2 = xsq + __shfl_xor(xsq, 32);
        if (hf == 0 && row0 + l32 < rows) sm.xn[l32] = xs2;
    }
    cn += __shfl_xor(cn, 32);
    __syncthreads();
    assign_finish<ID_BYTES, true>(B, P, sm, tot, (float)cn, col, row0);
}

// ============================================================ encode with a workspace
// With a caller's workspace an encode runs as (split_rows_kernel for fp32
// rows,) search_dots_kernel, decide_kernel, project_kernel: two plain bf16
// GEMMs whose tiles need not hold a row's whole search or residual, so that
// they can be cut to fill the chip, and one pass over the rows between them.
// A 1,560-row K + V chunk of bf16 rows (256 centers, r = 384): 18 + 15 + 24 us,
// the call 53.7 us, against 36 for assign_dma_kernel and 43 for
// encode_proj_kernel (98 and 196 blocks, which each stream the whole center
// table or a W_enc slice beside their rows; the call 76 us).  780 fp32 rows
// against 1,024 centers: 5 + 27 + 15 + 19 us (64 us a call) against 528 for
// assign_mfma_kernel (fp64) and 43 (571 us).  Bound by latency, not by a unit:
// project_kernel takes 8 us with one stage and 0.67 us per 128-wide stage (0.4
// of it LDS reads and writes at 128 B a cycle), search_dots_kernel 9 us with
// one stage.  Measured and not kept: four buffers of 64-wide stages (the same),
// eight (37 us: one block per CU), operand rows padded so that one k goes
// through all L2 channels (the same).

// GEMM core: acc += A[rows, K] B[cols, K]^T over stages [s0, s1) of KS k, up
// to two plane pairs one after the other.  Stages go global -> LDS by 1 KB DMA
// pieces into NBUF buffers, NBUF - 1 ahead, one barrier per stage.  A row of a
// stage is KS / 8 chunks of 16 bytes, chunk c of row q at slot c ^ swz(q): the
// 16 rows that one LDS cycle serves fall in 16 distinct slots.
template <int WM_, int WN_, int WR_, int WC_, int KS_, int NBUF_>
struct GemmTile {
    static constexpr int WM = WM_, WN = WN_, WR = WR_, WC = WC_, KS = KS_, NBUF = NBUF_;
    static constexpr int TM = 32 * WM * WR, TN = 32 * WN * WC, WAVES = WR * WC, THREADS = 64 * WAVES;
    static constexpr int ROWB = 2 * KS, CPR = KS / 8, RPP = 1024 / ROWB;   // bytes, chunks; rows per piece
    static constexpr int STAGE = (TM + TN) * ROWB, SMEM = NBUF * STAGE;
    // pieces e = wave + WAVES i: A's first, then B's; the first NHI waves take one more
    static constexpr int PA = TM / RPP, PIECES = (TM + TN) / RPP;
    static constexpr int QLO = PIECES / WAVES, NHI = PIECES % WAVES, QMAX = QLO + (NHI ? 1 : 0);
    static_assert(KS == 64 || KS == 128, "the swizzles below");
    static_assert(SMEM <= 160 * 1024, "LDS budget");
    static __device__ __forceinline__ int swz(int q) { return KS == 64 ? (q >> 1) & 7 : q & 15; }
    // row (of A's TM rows, then B's TN) that this lane brings in piece e
    static __device__ __forceinline__ int piece_row(int e) { return RPP * e + (threadIdx.x & 63) / CPR; }
    static __device__ __forceinline__ uint32_t piece_off(int q, int row, int64_t ld) {
        return (uint32_t)row * (uint32_t)(2 * ld) + 16 * (((threadIdx.x & 63) % CPR) ^ swz(q));
    }
};

// The second accumulators of a search: the first restart every SEG k, sums of
// squares of B's columns (of the first plane) beside them.
template <class T>
struct GemmTotals {
    f32x16 tot[T::WM][T::WN];
    float csq[T::WN], ctot[T::WN];
};

// spp stages of the operands' first planes, then of their second ones (a_plane
// and b_plane values on, 0: the same plane again); a at the tile's first row, b
// at the table, off this lane's byte offsets of its pieces.  SEG: see
// GemmTotals (0: none, t unused).
template <class T, int SEG>
__device__ __forceinline__ void gemm_stages(const uint16_t* a, int64_t a_plane, const uint16_t* b,
                                            int64_t b_plane, const uint32_t (&off)[T::QMAX], int s0,
                                            int s1, int spp, unsigned char* smem,
                                            f32x16 (&acc)[T::WM][T::WN], GemmTotals<T>& t, bool norms) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int hf = lane >> 5, l32 = lane & 31;
    const int wr = wave / T::WC, wc = wave % T::WC;
    auto issue = [&](int s) {
        const int p = s >= spp ? 1 : 0;
        const int64_t k = T::KS * (int64_t)(s - p * spp);
        const unsigned char* ab = reinterpret_cast<const unsigned char*>(a + p * a_plane + k);
        const unsigned char* bb = reinterpret_cast<const unsigned char*>(b + p * b_plane + k);
        unsigned char* dst = smem + ((s - s0) % T::NBUF) * T::STAGE;
#pragma unroll
        for (int i = 0; i < T::QMAX; ++i) {
            const int e = wave + T::WAVES * i;
            if (i < T::QLO || wave < T::NHI)
                dma16((e < T::PA ? ab + 0 : bb + 0) + off[i], dst + 1024 * e);
        }
    };
#pragma unroll
    for (int i = 0; i < T::NBUF - 1; ++i)
        if (s0 + i < s1) issue(s0 + i);
    for (int s = s0; s < s1; ++s) {
        // stage s landed; the NBUF - 2 after it may still be in flight
        if (s + T::NBUF - 2 >= s1) wait_vmcnt<0>();
        else if (T::NHI > 0 && wave < T::NHI) wait_vmcnt<(T::NBUF - 2) * T::QMAX>();
        else wait_vmcnt<(T::NBUF - 2) * T::QLO>();
        lds_barrier();
        if (s + T::NBUF - 1 < s1) issue(s + T::NBUF - 1);
        const unsigned char* sb = smem + ((s - s0) % T::NBUF) * T::STAGE;
#pragma unroll
        for (int k16 = 0; k16 < T::KS / 16; ++k16) {
            const int sw = 16 * ((2 * k16 + hf) ^ T::swz(l32));
            bf16x8 af[T::WM], bf[T::WN];
#pragma unroll
            for (int i = 0; i < T::WM; ++i)
                af[i] = lds_b128(reinterpret_cast<const uint16_t*>(
                    sb + (32 * (T::WM * wr + i) + l32) * T::ROWB + sw));
#pragma unroll
            for (int j = 0; j < T::WN; ++j)
                bf[j] = lds_b128(reinterpret_cast<const uint16_t*>(
                    sb + (T::TM + 32 * (T::WN * wc + j) + l32) * T::ROWB + sw));
#pragma unroll
            for (int i = 0; i < T::WM; ++i)
#pragma unroll
                for (int j = 0; j < T::WN; ++j) acc[i][j] = mfma32(af[i], bf[j], acc[i][j]);
            if constexpr (SEG > 0) {
                if (norms && s < spp) {
#pragma unroll
                    for (int j = 0; j < T::WN; ++j) {
                        const u32x4 v = __builtin_bit_cast(u32x4, bf[j]);
                        const uint32_t w4[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const bf16x2 wv = __builtin_bit_cast(bf16x2, w4[e]);
                            t.csq[j] = __builtin_amdgcn_fdot2_f32_bf16(wv, wv, t.csq[j], false);
                        }
                    }
                }
            }
        }
        if constexpr (SEG > 0) {
            if ((s - s0 + 1) % (SEG / T::KS) == 0 || s + 1 == s1) {
#pragma unroll
                for (int j = 0; j < T::WN; ++j) {
                    t.ctot[j] += t.csq[j];
                    t.csq[j] = 0.0f;
#pragma unroll
                    for (int i = 0; i < T::WM; ++i) {
#pragma unroll
                        for (int e = 0; e < 16; ++e) t.tot[i][j][e] += acc[i][j][e];
                        acc[i][j] = f32x16{};
                    }
                }
            }
        }
    }
}

// One problem's slices of the workspace.
struct EncWs {
    const uint16_t* xh;      // the rows' high plane [M][ld]: bf16 rows in place, or split
    const uint16_t* xl;      // low plane (fp32 rows), or NULL
    int64_t ld;
    float* dots;             // [splits][M][C rounded up to 4]
    float* cnorm;            // [splits][C]
    uint16_t* resid;         // [M][K]
};
struct EncWsBatch {
    EncBatch e;
    EncWs w[ENC_MAXB];
    int64_t m0;              // first row of this pass
    int rows;                // rows of the largest problem in this pass
    int splits;
};

// hi = bf16(x), lo = bf16(x - hi) of fp32 rows.
__global__ void __launch_bounds__(256) split_rows_kernel(EncWsBatch W) {
    const EncProb& P = W.e.p[blockIdx.y];
    const EncWs& w = W.w[blockIdx.y];
    const int per = W.e.K / 8;
    const int64_t n = (int64_t)min((int64_t)W.rows, P.M - W.m0) * per;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        const int64_t m = i / per;
        const int k = (int)(i - m * per) * 8;
        X8<false> x;
        x.load(P, W.m0 + m, k);
        u32x4 hi, lo;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            hi[e] = pack_bf16x2(x[2 * e], x[2 * e + 1]);
            lo[e] = pack_bf16x2(x[2 * e] - __uint_as_float(hi[e] << 16),
                                x[2 * e + 1] - __uint_as_float(hi[e] & 0xffff0000u));
        }
        *reinterpret_cast<u32x4*>(const_cast<uint16_t*>(w.xh) + m * w.ld + k) = hi;
        *reinterpret_cast<u32x4*>(const_cast<uint16_t*>(w.xl) + m * w.ld + k) = lo;
    }
}

// Approximate dot products of the search: split blockIdx.y of K's stages, rows
// and centers a 128 x 128 tile (32 x 64 per wave).  As in assign_bf16_kernel
// the MFMA accumulator restarts, here every SD_SEG k, and the segment sums are
// added in a second fp32 accumulator; the splits are added in fp64.  The
// blocks of the first row tile also sum ||c||^2 of their stages.
using DotsTile = GemmTile<1, 2, 4, 2, 64, 4>;
constexpr int SD_SEG = 128;

__global__ void __launch_bounds__(DotsTile::THREADS) search_dots_kernel(EncWsBatch W) {
    using T = DotsTile;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const EncProb& P = W.e.p[blockIdx.z];
    const EncWs& w = W.w[blockIdx.z];
    const int C = W.e.num_centers, K = W.e.K, spp = K / 64;
    const int nct = (C + T::TN - 1) / T::TN;
    const int tm0 = (int)(blockIdx.x / (uint32_t)nct) * T::TM;
    const int tn0 = (int)(blockIdx.x % (uint32_t)nct) * T::TN;
    const int left = (int)min(P.M - W.m0 - tm0, (int64_t)T::TM);
    if (left <= 0) return;
    const int total = w.xl ? 2 * spp : spp;
    const int s0 = (int)((uint32_t)total * blockIdx.y / (uint32_t)W.splits);
    const int s1 = (int)((uint32_t)total * (blockIdx.y + 1) / (uint32_t)W.splits);
    const uint16_t* xh = w.xh + tm0 * w.ld;
    uint32_t off[T::QMAX];
#pragma unroll
    for (int i = 0; i < T::QMAX; ++i) {
        const int e = (threadIdx.x >> 6) + T::WAVES * i, q = T::piece_row(e);
        off[i] = e < T::PA ? T::piece_off(q, min(q, left - 1), w.ld)
                           : T::piece_off(q, min(tn0 + q - T::TM, C - 1), K);
    }
    f32x16 acc[T::WM][T::WN] = {};
    GemmTotals<T> t = {};
    const bool norms = tm0 == 0;
    gemm_stages<T, SD_SEG>(xh, w.xl ? w.xl - w.xh : 0, P.centers, 0, off, s0, s1, spp, smem_raw, acc, t,
                           norms);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int hf = lane >> 5, l32 = lane & 31;
    const int wr = wave / T::WC, wc = wave % T::WC;
    const int Cs = (C + 3) & ~3;   // whole 16-byte pieces per row
    float* out = w.dots + (int64_t)blockIdx.y * W.rows * Cs;
#pragma unroll
    for (int j = 0; j < T::WN; ++j) {
        const int n = tn0 + 32 * (T::WN * wc + j) + l32;
        const float cn = t.ctot[j] + __shfl_xor(t.ctot[j], 32);
        if (n >= C) continue;
        if (norms && wr == 0 && hf == 0) w.cnorm[blockIdx.y * C + n] = cn;
#pragma unroll
        for (int i = 0; i < T::WM; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int m = 32 * (T::WM * wr + i) + 8 * (e / 4) + 4 * hf + (e % 4);
                if (m < left) out[(int64_t)(tm0 + m) * Cs + n] = t.tot[i][j][e];
            }
    }
}

// One wave per row: the search's decision (as assign_finish: U = min dt + E,
// candidates dt - E <= U, several compared exactly in fp64) and the bf16
// residual x - center - mean the projection reads.
// The bound: each segment's sum is within g_SEG of sum |x||c| of its k, the
// segment sums within g_n of theirs (n <= 96 segments per split), g_n = n 2^-24
// / (1 - n 2^-24); hi + lo misses 2^-16 |x|: (g_128 + g_96)(1 + 2^-7) + 2^-16
// < 2.9e-5 of ||x|| ||c|| per dot product, twice the rounding part if the
// matrix core truncated (4.3e-5).  ||c||^2 is summed the same way (< 1.4e-5
// ||c||^2).  The distance ||c||^2 - 2 x.c is then within 8.6e-5 ||x|| ||c|| +
// 2.8e-5 ||c||^2 of the exact one; E_c takes 1.2e-4 of both.
constexpr float SD_KAPPA = 1.2e-4f;
constexpr int SD_MAXC = 1024, SD_MAXK = 96 * SD_SEG / 2;

constexpr int DK_FLY = 6;   // 512-wide steps of a row in flight: 3,072 values

template <int ID_BYTES, bool XB, bool SEARCH>
__global__ void __launch_bounds__(256) decide_kernel(EncWsBatch W) {
    __shared__ float cns[SEARCH ? SD_MAXC : 1];
    const EncProb& P = W.e.p[blockIdx.y];
    const EncWs& w = W.w[blockIdx.y];
    const int t = threadIdx.x, lane = t & 63;
    const int C = W.e.num_centers, HD = W.e.K;
    const int64_t m = (int64_t)blockIdx.x * 4 + (t >> 6), gr = W.m0 + m;
    const bool row_ok = m < W.rows && gr < P.M;
    const int64_t cr_row = row_ok ? gr : 0;
    int id = 0;
    if constexpr (SEARCH) {
        for (int c = t; c < C; c += 256) {
            double cn = 0.0;
            for (int k = 0; k < W.splits; ++k) cn += (double)w.cnorm[k * C + c];
            cns[c] = (float)cn;
        }
        __syncthreads();
    }
    if (!row_ok) return;
    if constexpr (SEARCH) {
        constexpr int NQ = SD_MAXC / 256;
        // this lane's centers: 256 q + 4 lane + [0, 4); the splits' sums in fp64
        const int Cs = (C + 3) & ~3;
        const float* d = w.dots + m * Cs + 4 * lane;
        double dot[NQ][4] = {};
        for (int k = 0; k < W.splits; k += 2) {
            f32x4 v[2][NQ];
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int q = 0; q < NQ; ++q) {
                    v[u][q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                    if (256 * q + 4 * lane < C && k + u < W.splits)
                        v[u][q] = *reinterpret_cast<const f32x4*>(d + (int64_t)(k + u) * W.rows * Cs + 256 * q);
                }
#pragma unroll
            for (int q = 0; q < NQ; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) dot[q][e] += (double)v[0][q][e] + (double)v[1][q][e];
        }
        float xsq = 0.0f;
        for (int k0 = 8 * lane; k0 < HD; k0 += 512 * DK_FLY) {
            X8<XB> x[DK_FLY];
#pragma unroll
            for (int u = 0; u < DK_FLY; ++u)
                if (k0 + 512 * u < HD) x[u].load(P, cr_row, k0 + 512 * u);
#pragma unroll
            for (int u = 0; u < DK_FLY; ++u) {
                if (k0 + 512 * u >= HD) break;
#pragma unroll
                for (int e = 0; e < 8; ++e) xsq = fmaf(x[u][e], x[u][e], xsq);
            }
        }
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) xsq += __shfl_xor(xsq, off);
        const float xn = sqrtf(xsq) * 1.001f;
        float low[NQ][4];
        float U = INFINITY;
#pragma unroll
        for (int q = 0; q < NQ; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                low[q][e] = INFINITY;
                const int c = 256 * q + 4 * lane + e;
                if (c < C) {
                    const float cf = cns[c], dt = (float)((double)cf - 2.0 * dot[q][e]);
                    const float E = SD_KAPPA * (xn * sqrtf(cf) * 1.001f + cf * 1.001f);
                    low[q][e] = dt - E;
                    U = fminf(U, dt + E);
                }
            }
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) U = fminf(U, __shfl_xor(U, off));
        int cnt = 0, first = 0;
#pragma unroll
        for (int q = 0; q < NQ; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint64_t bits = __ballot(256 * q + 4 * lane + e < C && !(low[q][e] > U));
                if (bits) first = 256 * q + 4 * (__ffsll((unsigned long long)bits) - 1) + e;
                cnt += __popcll(bits);
            }
        // (overflowed sums and NaN: see assign_finish)
        const bool nan_row = xsq != xsq;
        id = nan_row ? 0 : first;
        if (cnt > 1 && !nan_row) {
            double bd = 0.0;
            int best = -1;
#pragma unroll
            for (int q = 0; q < NQ; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    uint64_t bits = __ballot(256 * q + 4 * lane + e < C && !(low[q][e] > U));
                    while (bits) {
                        const int c = 256 * q + 4 * (__ffsll((unsigned long long)bits) - 1) + e;
                        bits &= bits - 1;
                        const double dd = exact_distance<XB>(P, P.centers + (int64_t)c * HD, gr, HD, lane);
                        if (better(dd, c, bd, best) || (bd != bd && dd == dd)) { bd = dd; best = c; }
                    }
                }
            id = best;
        }
        if (lane == 0) store_id<ID_BYTES>(P.ids, gr, id);
    } else if (P.centers) {
        id = W.e.id_of(P, gr);
    }
    const uint16_t* cr = P.centers ? P.centers + (int64_t)id * HD : nullptr;
    for (int k0 = 8 * lane; k0 < HD; k0 += 512 * DK_FLY) {
        X8<XB> x[DK_FLY];
        u32x4 c[DK_FLY];
        f32x4 mn[DK_FLY][2];
#pragma unroll
        for (int u = 0; u < DK_FLY; ++u) {
            const int k = k0 + 512 * u;
            c[u] = u32x4{0, 0, 0, 0};
            mn[u][0] = mn[u][1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            if (k >= HD) continue;
            x[u].load(P, gr, k);
            if (cr) c[u] = *reinterpret_cast<const u32x4*>(cr + k);
            if (P.mean) {
                __builtin_memcpy(&mn[u][0], P.mean + k, 16);
                __builtin_memcpy(&mn[u][1], P.mean + k + 4, 16);
            }
        }
#pragma unroll
        for (int u = 0; u < DK_FLY; ++u) {
            if (k0 + 512 * u >= HD) break;
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const uint32_t cw = (e & 1) ? (c[u][e >> 1] & 0xffff0000u) : (c[u][e >> 1] << 16);
                // (x - 0 = x: absent centers or mean change nothing)
                v[e] = (x[u][e] - __uint_as_float(cw)) - mn[u][e >> 2][e & 3];
            }
            u32x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = pack_bf16x2(v[2 * e], v[2 * e + 1]);
            *reinterpret_cast<u32x4*>(w.resid + m * HD + k0 + 512 * u) = o;
        }
    }
}

// coeff = residual W_enc^T: one 32 x 32 accumulator per wave over the whole K
// in ascending steps of 16 (the bits of encode_proj_kernel), 64 rows x 64, 96
// or 128 columns per block.  Items (problem, row tile, column tile), column
// fastest, in one run per XCD: the column tiles of a row tile share its
// residual rows in one L2, W_enc (2.4 MB at r = 384) stays there.  Groups that
// divide the tile's columns are quantised here.
using Proj64 = GemmTile<1, 1, 2, 2, 128, 3>;
using Proj96 = GemmTile<1, 1, 2, 3, 128, 3>;
using Proj128 = GemmTile<1, 1, 2, 4, 64, 3>;

template <class T>
__global__ void __launch_bounds__(T::THREADS) project_kernel(EncWsBatch W) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int r = W.e.r, K = W.e.K;
    const uint32_t nct = (uint32_t)(r + T::TN - 1) / T::TN, nrt = (uint32_t)(W.rows + T::TM - 1) / T::TM;
    const uint32_t items = W.e.n * nrt * nct;
    const uint32_t item = (blockIdx.x & 7) * ((items + 7) >> 3) + (blockIdx.x >> 3);
    if (item >= items) return;
    const uint32_t rest = item / nct, prob = rest / nrt;
    const EncProb& P = W.e.p[prob];
    const EncWs& w = W.w[prob];
    const int tm0 = (int)(rest - prob * nrt) * T::TM, tn0 = (int)(item - rest * nct) * T::TN;
    const int left = (int)min(P.M - W.m0 - tm0, (int64_t)T::TM);
    if (left <= 0) return;
    const uint16_t* rs = w.resid + (int64_t)tm0 * K;
    uint32_t off[T::QMAX];
#pragma unroll
    for (int i = 0; i < T::QMAX; ++i) {
        const int e = (threadIdx.x >> 6) + T::WAVES * i, q = T::piece_row(e);
        off[i] = e < T::PA ? T::piece_off(q, min(q, left - 1), K)
                           : T::piece_off(q, min(tn0 + q - T::TM, r - 1), K);
    }
    f32x16 acc[1][1] = {};
    GemmTotals<T> none;
    gemm_stages<T, 0>(rs, 0, P.w_enc, 0, off, 0, K / T::KS, K / T::KS, smem_raw, acc, none, false);
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int hf = lane >> 5, l32 = lane & 31;
    const int n = tn0 + 32 * (wave % T::WC) + l32;
    const int64_t m0 = W.m0 + tm0;
    if (n < r) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int m = 32 * (wave / T::WC) + 8 * (e / 4) + 4 * hf + (e % 4);
            if (m < left) P.coeff[(m0 + m) * r + n] = acc[0][0][e];
        }
    }
    if (W.e.qgroup == 0) return;
    // the coefficients just stored, read back after the barrier
    __syncthreads();
    const int G = W.e.qgroup, ngroups = r / G, gpb = min(r - tn0, T::TN) / G, lpg = quant_lanes(G);
    for (int it0 = 0; it0 < T::TM * gpb; it0 += T::THREADS / lpg) {
        const int it = it0 + t / lpg;
        const bool in = it < T::TM * gpb && it / gpb < left;
        const int64_t gid = in ? (m0 + it / gpb) * ngroups + tn0 / G + it % gpb : P.M * ngroups;
        if (W.e.quant_mode == NKV_QUANT_BF16)
            quant_pack_group<NKV_QUANT_BF16>(P.coeff, P.M, r, G, W.e.scale_dtype, P.packed, P.scales, gid,
                                             t % lpg, lpg);
        else
            quant_pack_group<NKV_QUANT_FP32>(P.coeff, P.M, r, G, W.e.scale_dtype, P.packed, P.scales, gid,
                                             t % lpg, lpg);
    }
}

// ============================================================ MFMA GEMM core
// C[M, N] = A[M, K] * B[N, K]^T on v_mfma_f32_32x32x16_bf16.  A 256-thread
// block computes a 64 x 64 tile: wave w owns the 32 x 32 sub-tile
// (w / 2, w % 2).  K advances in steps of 32 through LDS.
//
// 32x32x16 operand layout (wave64): lane l supplies row (l % 32) of A and
// column (l % 32) of B, with k = 8 * (l / 32) + [0, 8) inside the 16-wide
// step.  The 16 accumulator values of lane l belong to column (l % 32) and
// rows 8 * (i / 4) + 4 * (l / 32) + (i % 4).
constexpr int GT_M = 64, GT_N = 64, GT_K = 32, GT_PAD = 8;

struct GemmSmem {
    uint16_t a[GT_M][GT_K + GT_PAD];
    uint16_t b[GT_N][GT_K + GT_PAD];
};

__device__ __forceinline__ bf16x8 lds_bf16x8(const uint16_t* p) {
    return *reinterpret_cast<const bf16x8*>(p);
}

// Encoder A-tile loader: A[m, k] = bf16(x[m, k] - center[id[m], k] - mean[k]).
struct EncodeA {
    const float* x;
    const uint16_t* centers;
    const void* ids;
    int id_bytes;
    int num_centers;
    const float* mean;
    int64_t M;
    int K;
    __device__ __forceinline__ int id_of(int64_t m) const {
        int v;
        if (id_bytes == 1) v = reinterpret_cast<const uint8_t*>(ids)[m];
        else if (id_bytes == 2) v = reinterpret_cast<const uint16_t*>(ids)[m];
        else v = reinterpret_cast<const int32_t*>(ids)[m];
        return min(max(v, 0), num_centers - 1);
    }
    // thread t fills row t/4, k-columns (t%4)*8 .. +8 of the 64 x 32 tile
    __device__ __forceinline__ void load(GemmSmem& s, int64_t m0, int k0, int t) const {
        const int rr = t / 4, kc = (t % 4) * 8;
        const int64_t m = m0 + rr;
        u32x4 packedv = {0, 0, 0, 0};
        if (m < M) {
            const float* xp = x + m * K + k0 + kc;
            f32x4 x0 = *reinterpret_cast<const f32x4*>(xp);
            f32x4 x1 = *reinterpret_cast<const f32x4*>(xp + 4);
            float v[8] = {x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
            if (centers) {
                const uint16_t* cp = centers + (int64_t)id_of(m) * K + k0 + kc;
                u32x4 cw = *reinterpret_cast<const u32x4*>(cp);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    v[2 * e] = v[2 * e] - __uint_as_float(cw[e] << 16);
                    v[2 * e + 1] = v[2 * e + 1] - __uint_as_float(cw[e] & 0xffff0000u);
                }
            }
            if (mean) {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = v[e] - mean[k0 + kc + e];
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) packedv[e] = pack_bf16x2(v[2 * e], v[2 * e + 1]);
        }
        *reinterpret_cast<u32x4*>(&s.a[rr][kc]) = packedv;
    }
};

// Decoder A-tile loader: A[m, k] = bf16(code * scale) of row src(m).
struct DecodeA {
    const uint8_t* packed;
    const uint16_t* scales;
    const int32_t* row_index;
    int scale_dtype;
    int group;
    int64_t M;   // output rows
    int K;       // r
    __device__ __forceinline__ void load(GemmSmem& s, int64_t m0, int k0, int t) const {
        const int rr = t / 4, kc = (t % 4) * 8;
        const int64_t m = m0 + rr;
        u32x4 o = {0, 0, 0, 0};
        if (m < M) {
            const int64_t src = row_index ? (int64_t)row_index[m] : m;
            const uint32_t word =
                *reinterpret_cast<const uint32_t*>(packed + src * (K / 2) + (k0 + kc) / 2);
            const float sc =
                scale_bits_to_f32(scales[src * (K / group) + (k0 + kc) / group], scale_dtype);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float lo = (float)((int)((word >> (8 * e)) & 15u) - 7) * sc;
                float hi = (float)((int)((word >> (8 * e + 4)) & 15u) - 7) * sc;
                o[e] = pack_bf16x2(lo, hi);
            }
        }
        *reinterpret_cast<u32x4*>(&s.a[rr][kc]) = o;
    }
};

// B tile [64 rows (n) x 32 k] of a bf16 row-major [N, K] matrix.
__device__ __forceinline__ void load_b_tile(GemmSmem& s, const uint16_t* __restrict__ B,
                                            int64_t N, int K, int64_t n0, int k0, int t) {
    const int rr = t / 4, kc = (t % 4) * 8;
    const int64_t n = n0 + rr;
    u32x4 v = {0, 0, 0, 0};
    if (n < N) v = *reinterpret_cast<const u32x4*>(B + n * K + k0 + kc);
    *reinterpret_cast<u32x4*>(&s.b[rr][kc]) = v;
}

template <class ALoader>
__device__ __forceinline__ f32x16 gemm_tile(GemmSmem& s, const ALoader& al,
                                            const uint16_t* __restrict__ B, int64_t N, int K,
                                            int64_t m0, int64_t n0) {
    const int t = threadIdx.x;
    const int lane = t & 63, wave = t >> 6;
    const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
    const int hf = lane >> 5, l32 = lane & 31;
    f32x16 acc = {};
    for (int k0 = 0; k0 < K; k0 += GT_K) {
        __syncthreads();
        al.load(s, m0, k0, t);
        load_b_tile(s, B, N, K, n0, k0, t);
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < GT_K; kk += 16) {
            bf16x8 a = lds_bf16x8(&s.a[wm + l32][kk + 8 * hf]);
            bf16x8 b = lds_bf16x8(&s.b[wn + l32][kk + 8 * hf]);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
        }
    }
    return acc;
}

__global__ void __launch_bounds__(256) encode_gemm_kernel(EncodeA al,
                                                          const uint16_t* __restrict__ w_enc,
                                                          int r, float* __restrict__ coeff) {
    __shared__ GemmSmem s;
    const int64_t m0 = (int64_t)blockIdx.x * GT_M, n0 = (int64_t)blockIdx.y * GT_N;
    f32x16 acc = gemm_tile(s, al, w_enc, r, al.K, m0, n0);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int hf = lane >> 5, l32 = lane & 31;
    const int64_t n = n0 + (wave & 1) * 32 + l32;
    if (n >= r) return;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int64_t m = m0 + (wave >> 1) * 32 + 8 * (i / 4) + 4 * hf + (i % 4);
        if (m < al.M) coeff[m * r + n] = acc[i];
    }
}

// Encoder projection coeff[M, r] = bf16(x - center[id] - mean) W_enc^T, fp32
// accumulation (MG nanokv_codec.py:344-347: the residual minus the mean, in
// bf16, through the bf16 operator).  A block of six waves owns 32 rows x 192
// coefficient columns (wave w: columns 32w .. 32w + 32) and walks K in
// 128-wide stages.  Every operand goes global -> LDS by 1 KB DMA pieces,
// double-buffered (no register staging, so no wait covers more than the
// stage it needs):
//   [W_enc 192 rows x 256 B][inputs 32 rows][center values 32 rows][mean]
// (the mean piece holds the stage's 128 means twice).  Stage i: wait, barrier,
// issue stage i + 1, waves 0-3 turn stage i into the bf16 residual image (two
// 16-byte units of one row per thread), barrier, 8 MFMAs per wave.  A block's
// stream is bound by a fixed cost per barrier plus one per piece, so few
// large stages stream faster than many small ones (64-wide stages four deep
// took 34.5-39.6 us for a 1,560-row K+V chunk).  W and the residual image are
// [row][16 chunks of 16 bytes] with chunk c of row q at slot c ^ (q % 8), so
// the operand reads (32 rows at one chunk) are free of bank conflicts.  Needs
// K % 128 == 0 and 16-byte aligned rows.
constexpr int EP_ROWS = 32, EP_WAVES = 6, EP_COLS = 32 * EP_WAVES, EP_KS = 128;
constexpr int EP_CPR = EP_KS / 8;                  // 16-byte chunks per bf16 row
constexpr int EP_RPP = 1024 / (EP_KS * 2);         // bf16 rows per 1 KB piece
constexpr int EP_WPIECES = EP_COLS / EP_RPP;

template <bool XB>
struct EncProjFmt {
    static constexpr int XROW = EP_KS * (XB ? 2 : 4);               // input bytes per row
    static constexpr int XPIECES = EP_ROWS * XROW / 1024;
    static constexpr int X0 = EP_WPIECES, C0 = X0 + XPIECES, M0 = C0 + EP_ROWS / EP_RPP;
    static constexpr int PIECES = M0 + 1;
    static constexpr int STAGE = PIECES * 1024;                      // bytes
    static constexpr int AIMG = EP_ROWS * EP_KS * 2;                 // residual image bytes
    static constexpr int SMEM = 2 * STAGE + AIMG;
    // pieces per wave and stage: the first PIECES % EP_WAVES waves take one more
    static constexpr int QLO = PIECES / EP_WAVES, NHI = PIECES % EP_WAVES;
    static constexpr int QMAX = QLO + (NHI ? 1 : 0);
};

template <bool XB>
__global__ void __launch_bounds__(64 * EP_WAVES) encode_proj_kernel(EncBatch B) {
    using F = EncProjFmt<XB>;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    // items: (problem, column slice, row block), row block fastest
    const int ncb = (B.r + EP_COLS - 1) / EP_COLS;
    const int64_t item = xcd_item(blockIdx.x, B.n * ncb * B.row_blocks);
    if (item >= B.n * ncb * B.row_blocks) return;
    const int64_t rest = item / B.row_blocks;
    const EncProb& P = B.p[rest / ncb];
    const int r = B.r, K = B.K, S = K / EP_KS;
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int hf = lane >> 5, l32 = lane & 31;
    const int64_t m0 = (item % B.row_blocks) * EP_ROWS;
    if (m0 >= P.M) return;
    const int n0 = (int)(rest % ncb) * EP_COLS;
    // this wave's pieces e = wave + EP_WAVES i: per lane a source address
    // and the bytes it advances per stage.  Rows past the end read the last
    // row; absent centers or mean read W_enc (any readable bytes; unused).
    const unsigned char* src[F::QMAX];
    int64_t adv[F::QMAX];
    auto xrow = [&](int q) { return min(m0 + q, P.M - 1); };
#pragma unroll
    for (int i = 0; i < F::QMAX; ++i) {
        const int e = wave + EP_WAVES * i;
        const unsigned char* sp = reinterpret_cast<const unsigned char*>(P.w_enc);
        int64_t st = 0;
        if (e < F::X0) {
            // W row n0 + q, slot lane % EP_CPR holds chunk slot ^ (q % 8)
            const int q = EP_RPP * e + lane / EP_CPR;
            const int row = min(n0 + q, r - 1);
            sp = reinterpret_cast<const unsigned char*>(P.w_enc + (int64_t)row * K +
                                                        8 * ((lane % EP_CPR) ^ (q & 7)));
            st = 2 * EP_KS;
        } else if (e < F::C0) {
            constexpr int CPRX = F::XROW / 16, RPPX = 1024 / F::XROW;
            const int64_t m = xrow(RPPX * (e - F::X0) + lane / CPRX);
            const int off = 16 * (lane % CPRX);
            sp = XB ? reinterpret_cast<const unsigned char*>(P.xb + m * P.ldx) + off
                    : reinterpret_cast<const unsigned char*>(P.x + m * P.ldx) + off;
            st = F::XROW;
        } else if (e < F::M0) {
            if (P.centers) {
                const int64_t m = xrow(EP_RPP * (e - F::C0) + lane / EP_CPR);
                sp = reinterpret_cast<const unsigned char*>(P.centers + (int64_t)B.id_of(P, m) * K +
                                                            8 * (lane % EP_CPR));
                st = 2 * EP_KS;
            }
        } else if (e == F::M0) {
            if (P.mean) {
                sp = reinterpret_cast<const unsigned char*>(P.mean + 4 * (lane % (EP_KS / 4)));
                st = 4 * EP_KS;
            }
        }
        src[i] = sp;
        adv[i] = st;
    }
    auto issue = [&](int stg) {
        unsigned char* dst = smem_raw + (stg & 1) * F::STAGE;
#pragma unroll
        for (int i = 0; i < F::QMAX; ++i) {
            const int e = wave + EP_WAVES * i;
            if (i < F::QLO || wave < F::NHI) dma16(src[i] + stg * adv[i], dst + 1024 * e);
        }
    };
    unsigned char* aimg = smem_raw + 2 * F::STAGE;
    const bool prod = wave < 4;
    // stage stg (landed) -> the residual image; absent centers or mean
    // subtract zeros (x - 0 = x exactly), so every read is unconditional
    const bool has_c = P.centers != nullptr, has_m = P.mean != nullptr;
    auto prep = [&](int stg) {
        const unsigned char* sb = smem_raw + (stg & 1) * F::STAGE;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int unit = t + 256 * u;                       // of 32 rows x 16 chunks
            const int arow = unit / EP_CPR, ach = unit % EP_CPR;
            const u32x4 c = *reinterpret_cast<const u32x4*>(sb + 1024 * F::C0 + arow * (EP_KS * 2) + 16 * ach);
            const f32x4* mp = reinterpret_cast<const f32x4*>(sb + 1024 * F::M0 + 32 * ach);
            const f32x4 u0 = mp[0], u1 = mp[1];
            float xv[8];
            if constexpr (XB) {
                const u32x4 w = *reinterpret_cast<const u32x4*>(sb + 1024 * F::X0 + arow * F::XROW + 16 * ach);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    xv[2 * e] = __uint_as_float(w[e] << 16);
                    xv[2 * e + 1] = __uint_as_float(w[e] & 0xffff0000u);
                }
            } else {
                const f32x4* xp = reinterpret_cast<const f32x4*>(sb + 1024 * F::X0 + arow * F::XROW + 32 * ach);
                const f32x4 a0 = xp[0], a1 = xp[1];
#pragma unroll
                for (int e = 0; e < 4; ++e) { xv[e] = a0[e]; xv[4 + e] = a1[e]; }
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const uint32_t cw = (e & 1) ? (c[e >> 1] & 0xffff0000u) : (c[e >> 1] << 16);
                const float cv = has_c ? __uint_as_float(cw) : 0.0f;
                const float mv = has_m ? (e < 4 ? u0[e] : u1[e - 4]) : 0.0f;
                xv[e] = (xv[e] - cv) - mv;
            }
            const bool ok = m0 + arow < P.M;
            u32x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = ok ? pack_bf16x2(xv[2 * e], xv[2 * e + 1]) : 0u;
            *reinterpret_cast<u32x4*>(aimg + arow * (EP_KS * 2) + 16 * (ach ^ (arow & 7))) = o;
        }
    };
    const bool cols = n0 + 32 * wave < r;
    f32x16 acc = {};
    const int arow_b = l32 * (EP_KS * 2), wrow_b = (32 * wave + l32) * (EP_KS * 2);
    auto compute = [&](int stg) {
        const unsigned char* wr = smem_raw + (stg & 1) * F::STAGE + wrow_b;
        bf16x8 af[EP_KS / 16], wf[EP_KS / 16];
#pragma unroll
        for (int k16 = 0; k16 < EP_KS / 16; ++k16) {
            const int slot = 16 * ((2 * k16 + hf) ^ (l32 & 7));
            af[k16] = lds_b128(reinterpret_cast<const uint16_t*>(aimg + arow_b + slot));
            wf[k16] = lds_b128(reinterpret_cast<const uint16_t*>(wr + slot));
        }
        // all reads in flight before the first product
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k16 = 0; k16 < EP_KS / 16; ++k16)
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[k16], wf[k16], acc, 0, 0, 0);
    };
    issue(0);
    for (int it = 0; it < S; ++it) {
        // stage it landed (nothing later is in flight yet); after the barrier
        // every wave is past stage it - 1, whose buffer takes stage it + 1
        wait_vmcnt<0>();
        lds_barrier();
        if (it + 1 < S) issue(it + 1);
        if (prod) prep(it);
        lds_barrier();
        if (cols) compute(it);
    }
    const int n = n0 + 32 * wave + l32;
    if (cols && n < r) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int64_t mm = m0 + 8 * (i / 4) + 4 * hf + (i % 4);
            if (mm < P.M) P.coeff[mm * r + n] = acc[i];
        }
    }
    if (B.qgroup == 0) return;
    // the quantiser on the block's whole groups (the columns of a block hold
    // whole groups): the coefficients just stored, read back after the barrier
    __syncthreads();
    const int G = B.qgroup, ngroups = r / G, gpb = (min(r - n0, EP_COLS)) / G;
    const int lpg = quant_lanes(G);
    for (int it0 = 0; it0 < EP_ROWS * gpb; it0 += 64 * EP_WAVES / lpg) {
        const int it = it0 + t / lpg;
        // (groups past the block's last: out of range, like rows past the end)
        const int64_t gid = it < EP_ROWS * gpb ? (m0 + it / gpb) * ngroups + n0 / G + it % gpb
                                               : P.M * ngroups;
        if (B.quant_mode == NKV_QUANT_BF16)
            quant_pack_group<NKV_QUANT_BF16>(P.coeff, P.M, r, G, B.scale_dtype, P.packed, P.scales, gid,
                                             t % lpg, lpg);
        else
            quant_pack_group<NKV_QUANT_FP32>(P.coeff, P.M, r, G, B.scale_dtype, P.packed, P.scales, gid,
                                             t % lpg, lpg);
    }
}

static_assert(EncProjFmt<false>::SMEM <= 160 * 1024, "LDS budget");

struct DecodeEpi {
    const uint16_t* centers;   // [C, HD] for this batch item, or NULL
    const void* ids;           // [N] of this batch item
    int id_bytes;
    int num_centers;
    const int32_t* row_index;
    const float* mean;
    // ids outside the table are clamped (a corrupt payload must not read out of bounds)
    __device__ __forceinline__ int id_of(int64_t src) const {
        int v;
        if (id_bytes == 1) v = reinterpret_cast<const uint8_t*>(ids)[src];
        else if (id_bytes == 2) v = reinterpret_cast<const uint16_t*>(ids)[src];
        else v = reinterpret_cast<const int32_t*>(ids)[src];
        return min(max(v, 0), num_centers - 1);
    }
};

// out[m, n] = bf16(bf16(acc + bf16(mean[n])) + center[id[src(m)], n])   (MG:438-454)
__global__ void __launch_bounds__(256) decode_gemm_kernel(DecodeA al, DecodeEpi ep,
                                                          const uint16_t* __restrict__ w_dec,
                                                          int HD, uint16_t* __restrict__ out) {
    __shared__ GemmSmem s;
    const int64_t m0 = (int64_t)blockIdx.x * GT_M, n0 = (int64_t)blockIdx.y * GT_N;
    f32x16 acc = gemm_tile(s, al, w_dec, HD, al.K, m0, n0);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int hf = lane >> 5, l32 = lane & 31;
    const int64_t n = n0 + (wave & 1) * 32 + l32;
    if (n >= HD) return;
    const float bias = ep.mean ? bf16_round(ep.mean[n]) : 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int64_t m = m0 + (wave >> 1) * 32 + 8 * (i / 4) + 4 * hf + (i % 4);
        if (m >= al.M) continue;
        float v = bf16_round(acc[i] + bias);
        if (ep.centers) {
            const int64_t src = ep.row_index ? (int64_t)ep.row_index[m] : m;
            v = bf16_round(v + bf16_bits_to_f32(ep.centers[(int64_t)ep.id_of(src) * HD + n]));
        }
        out[m * HD + n] = f32_to_bf16_bits(v);
    }
}


// ============================================================ staged decode
// out[m, n] = bf16(bf16(latent[m] . w_dec[n] + bf16(mean[n])) + center[id[m], n])
// (MG:438-454) for up to DEC_MAXB problems of one shape in one launch: the
// segments of a cache, batch items.  A block owns 32 MI WR rows x 64 WC
// columns (wave (wr, wc): 32 MI rows x 64 columns) and walks r in 64-wide
// slices:
//   - W_dec slice [columns][64] by 1 KB DMA pieces, double-buffered, issued
//     one slice ahead;
//   - the codes of the slice, held in registers one slice ahead (16 per
//     thread), unpacked once per block into the latent image [rows][64].
// Both images are [row][8 chunks of 16 bytes] with chunk c of row q at slot
// c ^ ((q >> 1) & 7): the 16 rows that one LDS cycle serves fall in 16
// distinct slots.  W is the MFMA's row operand, so a lane ends with four
// consecutive columns of one row; bf16(acc + mean) goes through LDS and out
// as whole 16-byte pieces of rows, the center row's piece added on the way.
// The accumulator takes k in ascending steps of 16, as decode_gemm_kernel
// does: the same bits.
// Measured (12,480 x 3,072, r = 384, centers): 52.7 us = 559 TFLOP/s, 1.5 TB/s
// written, against 214 us for decode_gemm_kernel (one 64 x 64 tile per block,
// codes unpacked per 64 columns, 2-byte stores) and 43 us more to concatenate
// the segments.  Not bound by one unit: with the W copies, the unpack or the
// MFMAs left out it takes 47, 43 and 39 us; the rest (output, centers) 17.
constexpr int DEC_MAXB = 16, DT_K = 64;
struct DecProb {
    const uint8_t* packed;
    const uint16_t* scales;
    const void* ids;
    const uint16_t* centers;   // [C, HD], or NULL
    const int32_t* row_index;  // [M], or NULL
    uint16_t* out;             // [M, HD]
    int64_t M;
    int id_bytes, num_centers;
};
struct DecBatch {
    DecProb p[DEC_MAXB];
    const uint16_t* w;         // [HD, r]
    const float* mean;         // [HD], or NULL
    int n, HD, r, group, scale_dtype;
    uint32_t row_blocks;       // of the largest problem
};

// bf16((code - 7) * scale) of eight codes, as unpack_kernel forms it (the
// one-fma form of unpack8 gives NaN where an infinite scale gives +-inf here).
__device__ __forceinline__ u32x4 latent8(uint32_t w, float s) {
    uint32_t ev = w & 0x0f0f0f0fu, od = (w >> 4) & 0x0f0f0f0fu;
    asm("" : "+v"(ev));  // one v_cvt_f32_ubyte per code (see unpack8)
    asm("" : "+v"(od));
    u32x4 o;
#pragma unroll
    for (int b = 0; b < 4; ++b)
        o[b] = pack_bf16x2(((float)((ev >> (8 * b)) & 0xffu) - 7.0f) * s,
                           ((float)((od >> (8 * b)) & 0xffu) - 7.0f) * s);
    return o;
}

template <int MI, int WR, int WC>
struct DecFmt {
    static constexpr int ROWS = 32 * MI * WR, COLS = 64 * WC, WAVES = WR * WC, THREADS = 64 * WAVES;
    static constexpr int WSTAGE = COLS * DT_K * 2, AIMG = ROWS * DT_K * 2;
    static constexpr int WPIECES = WSTAGE / 1024 / WAVES;      // DMA pieces per wave
    static constexpr int OSTRIDE = COLS * 2 + 16;              // staged output row, bytes
    static constexpr int CROW = ROWS * OSTRIDE;                // center row pointers, after the GEMM
    static constexpr int SMEM = 2 * WSTAGE + AIMG;
    static_assert(CROW + 8 * ROWS <= SMEM, "the output tile fits the GEMM's buffers");
    static constexpr bool BIG = MI == 2;
    static constexpr int UNITS = ROWS * COLS / 8 / THREADS;    // 16-byte output pieces per thread
    static_assert(ROWS * 4 == THREADS, "a thread unpacks 16 codes of one row");
    static_assert(WSTAGE % (1024 * WAVES) == 0, "whole pieces per wave");
};

template <int MI, int WR, int WC>
__global__ void __launch_bounds__(64 * WR * WC, 4) decode_tile_kernel(DecBatch B) {
    using F = DecFmt<MI, WR, WC>;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    // items: (problem, row block, column block), column block fastest, eight
    // equal runs, one per XCD: the blocks of one XCD share code and center rows
    const uint32_t ncb = (uint32_t)(B.HD + F::COLS - 1) / F::COLS;
    const uint32_t items = (uint32_t)B.n * B.row_blocks * ncb;
    const uint32_t item = (blockIdx.x & 7) * ((items + 7) >> 3) + (blockIdx.x >> 3);
    if (item >= items) return;
    const uint32_t rest = item / ncb, prob = rest / B.row_blocks;
    const DecProb& P = B.p[prob];
    const int64_t m0 = (int64_t)(rest - prob * B.row_blocks) * F::ROWS;
    if (m0 >= P.M) return;
    const int n0 = (int)(item - rest * ncb) * F::COLS;
    const int r = B.r, S = (r + DT_K - 1) / DT_K;
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int hf = lane >> 5, l32 = lane & 31;
    const int wr = wave / WC, wc = wave % WC;
    // this thread's codes: row t / 4, k 16 (t % 4) .. +16 of each slice
    const int arow = t >> 2, aq = t & 3;
    int64_t src = min(m0 + arow, P.M - 1);
    if (P.row_index) src = P.row_index[src];
    const uint8_t* cp = P.packed + src * (r / 2) + 8 * aq;
    const uint16_t* sp = P.scales + src * (r / B.group);
    const uint16_t* my_crow = nullptr;
    if (P.centers && aq == 0) {
        const int id = min(max(read_id(P.ids, P.id_bytes, src), 0), P.num_centers - 1);
        my_crow = P.centers + (int64_t)id * B.HD;
    }
    const float inv_g = 1.0f / (float)B.group;
    // floor(k / group) for k < 2^20: (k + 0.5) / group is at least 0.5 / group
    // from an integer, the product's error is below k 2^-22 / group
    auto grp = [&](int k) { return (int)(((float)k + 0.5f) * inv_g); };
    // W pieces: piece e = wave + WAVES i holds columns 8e .. 8e + 8 (pieces
    // past HD: the last eight); lane L brings slot L % 8 of column 8e + L / 8.
    // WAVES is even, so the slot's chunk is the same in every piece.  A half
    // slice (r % 64 == 32) repeats its first half in the second; unused.
    static_assert(F::WAVES % 2 == 0, "one lane offset serves every piece");
    const int wq = 8 * wave + (lane >> 3), wch = (lane & 7) ^ ((wq >> 1) & 7);
    const uint32_t woff = (uint32_t)(lane >> 3) * (uint32_t)(2 * r);
    const uint32_t woff_full = woff + 16 * wch, woff_half = woff + 16 * (wch & 3);
    auto issue_w = [&](int s) {
        unsigned char* dst = smem_raw + (s & 1) * F::WSTAGE;
        const uint32_t off = r - s * DT_K >= DT_K ? woff_full : woff_half;
#pragma unroll
        for (int i = 0; i < F::WPIECES; ++i) {
            const int e = wave + F::WAVES * i;
            const unsigned char* g = reinterpret_cast<const unsigned char*>(B.w) +
                                     2 * ((int64_t)min(n0 + 8 * e, B.HD - 8) * r + s * DT_K);
            dma16(g + off, dst + 1024 * e);
        }
    };
    u32x2 code;
    float sc[2];
    const bool g16 = B.group % 16 == 0;
    auto load_codes = [&](int s) {
        const int k = s * DT_K + 16 * aq;
        if (k < r) {
            code = *reinterpret_cast<const u32x2*>(cp + s * (DT_K / 2));
            sc[0] = sc[1] = scale_bits_to_f32(sp[grp(k)], B.scale_dtype);
            if (!g16) sc[1] = scale_bits_to_f32(sp[grp(k + 8)], B.scale_dtype);
        }
    };
    unsigned char* aimg = smem_raw + 2 * F::WSTAGE;
    const int asw = (arow >> 1) & 7;
    f32x16 acc[MI][2] = {};
    issue_w(0);
    load_codes(0);
    for (int s = 0; s < S; ++s) {
        const int kn = min(r - s * DT_K, DT_K);
        if (16 * aq < kn) {
#pragma unroll
            for (int c = 0; c < 2; ++c)
                *reinterpret_cast<u32x4*>(aimg + arow * (DT_K * 2) + 16 * ((2 * aq + c) ^ asw)) =
                    latent8(code[c], sc[c]);
        }
        // slice s landed and its latent image is written (nothing later is in flight)
        wait_vmcnt<0>();
        lds_barrier();
        if (s + 1 < S) {
            issue_w(s + 1);
            load_codes(s + 1);
        }
        const unsigned char* wb = smem_raw + (s & 1) * F::WSTAGE;
#pragma unroll
        for (int k16 = 0; k16 < DT_K / 16; ++k16) {
            if (16 * k16 >= kn) break;
            const int sw = 16 * ((2 * k16 + hf) ^ ((l32 >> 1) & 7));
            bf16x8 wf[2], af[MI];
#pragma unroll
            for (int j = 0; j < 2; ++j)
                wf[j] = lds_b128(reinterpret_cast<const uint16_t*>(
                    wb + (64 * wc + 32 * j + l32) * (DT_K * 2) + sw));
#pragma unroll
            for (int i = 0; i < MI; ++i)
                af[i] = lds_b128(reinterpret_cast<const uint16_t*>(
                    aimg + (32 * (MI * wr + i) + l32) * (DT_K * 2) + sw));
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[i][j] = mfma32(wf[j], af[i], acc[i][j]);
        }
        lds_barrier();
    }
    const uint16_t** crow = reinterpret_cast<const uint16_t**>(smem_raw + F::CROW);
    if (aq == 0) crow[arow] = my_crow;
    // bf16(acc + mean) to LDS: lane (hf, l32) holds row l32 of its tiles,
    // columns 8 q + 4 hf + [0, 4) for q = 0 .. 3
    const int nl = 64 * wc + 4 * hf;
    f32x4 mean[8];
#pragma unroll
    for (int jq = 0; jq < 8; ++jq) {
        mean[jq] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        if (B.mean) {
            __builtin_memcpy(&mean[jq], B.mean + min(n0 + nl + 8 * jq, B.HD - 4), 16);
        }
    }
#pragma unroll
    for (int jq = 0; jq < 8; ++jq) {
#pragma unroll
        for (int e = 0; e < 4; ++e) mean[jq][e] = bf16_round(mean[jq][e]);
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            const f32x16& v = acc[i][jq >> 2];
            u32x2 o;
#pragma unroll
            for (int e = 0; e < 2; ++e)
                o[e] = pack_bf16x2(v[4 * (jq & 3) + 2 * e] + mean[jq][2 * e],
                                   v[4 * (jq & 3) + 2 * e + 1] + mean[jq][2 * e + 1]);
            *reinterpret_cast<u32x2*>(smem_raw + (32 * (MI * wr + i) + l32) * F::OSTRIDE +
                                      2 * (nl + 8 * jq)) = o;
        }
    }
    __syncthreads();
    // out: consecutive threads take consecutive 16-byte pieces of a row
    constexpr int CH = F::COLS / 8, RSTEP = F::THREADS / CH;
    const int frow = t / CH, fch = t % CH, n = n0 + 8 * fch;
    if (n >= B.HD) return;
    const int rows = (int)min(P.M - m0, (int64_t)F::ROWS);
    uint16_t* out = P.out + (m0 + frow) * B.HD + n;
    const unsigned char* st = smem_raw + frow * F::OSTRIDE + 16 * fch;
    // a large output (16 MB and more) streams past the L2, which then keeps
    // W_dec and the centers: 56.5 -> 52.7 us for 12,480 x 3,072 at r = 384
    auto put = [&](int u, const u32x4& v) {
        u32x4* o = reinterpret_cast<u32x4*>(out + (int64_t)RSTEP * u * B.HD);
        if constexpr (F::BIG) __builtin_nontemporal_store(v, o);
        else *o = v;
    };
    if (P.centers) {
        u32x4 cv[F::UNITS];   // rows past the end have the last row's center
#pragma unroll
        for (int u = 0; u < F::UNITS; ++u)
            cv[u] = ldg(reinterpret_cast<const u32x4*>(crow[frow + RSTEP * u] + n));
#pragma unroll
        for (int u = 0; u < F::UNITS; ++u) {
            u32x4 v = *reinterpret_cast<const u32x4*>(st + RSTEP * u * F::OSTRIDE);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                v[e] = pack_bf16x2(__uint_as_float(v[e] << 16) + __uint_as_float(cv[u][e] << 16),
                                   __uint_as_float(v[e] & 0xffff0000u) +
                                       __uint_as_float(cv[u][e] & 0xffff0000u));
            if (frow + RSTEP * u < rows) put(u, v);
        }
    } else {
#pragma unroll
        for (int u = 0; u < F::UNITS; ++u)
            if (frow + RSTEP * u < rows)
                put(u, *reinterpret_cast<const u32x4*>(st + RSTEP * u * F::OSTRIDE));
    }
}

using DecBig = DecFmt<2, 2, 4>;
using DecSmall = DecFmt<1, 2, 2>;
static_assert(2 * DecBig::SMEM <= 160 * 1024, "two blocks per CU");

}  // namespace nkv

using namespace nkv;

// ============================================================ C ABI
static int check_codec_layout(int r, int group, int scale_dtype) {
    NKV_REQUIRE(r > 0 && r % 32 == 0, NKV_ERR_INVALID, "r must be a positive multiple of 32");
    NKV_REQUIRE(group > 0 && r % group == 0 && group % 8 == 0, NKV_ERR_INVALID,
                "group must divide r and be a multiple of 8");
    NKV_REQUIRE(scale_dtype == NKV_DTYPE_BF16 || scale_dtype == NKV_DTYPE_FP16,
                NKV_ERR_INVALID, "scale_dtype must be NKV_DTYPE_BF16 or NKV_DTYPE_FP16");
    return NKV_OK;
}

namespace nkv {

// ------------------------------------------------------- INT8 operator weights
// _pack_operator (MG:108-131): per (row, group) s = max(amax|w|, 1e-12) / 127
// in fp32, q = clamp(rint(w / s), -127, 127), stored scale = bf16(s) (the codes
// use the unrounded s).  One wave per (row, group): a wave-wide amax, then
// every lane codes elements lane, lane + 64, ...
__global__ void __launch_bounds__(256) int8_pack_kernel(const float* __restrict__ w, int64_t rows,
                                                        int cols, int group,
                                                        int8_t* __restrict__ q,
                                                        uint16_t* __restrict__ scale) {
    const int lane = threadIdx.x & 63;
    const int ngroups = cols / group;
    const int64_t gid = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (gid >= rows * ngroups) return;  // uniform per wave
    const int64_t row = gid / ngroups;
    const int64_t base = row * cols + (gid - row * ngroups) * (int64_t)group;
    float amax = 0.0f;
    for (int j = lane; j < group; j += 64) {
        const float a = fabsf(w[base + j]);
        amax = (a > amax || a != a) ? a : amax;  // NaN propagates like torch.amax
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const float b = __shfl_xor(amax, o);
        amax = (b > amax || b != b) ? b : amax;
    }
    const float s = __fdiv_rn((amax > 1e-12f || amax != amax) ? amax : 1e-12f, 127.0f);
    if (lane == 0) scale[gid] = f32_to_bf16_bits(s);
    for (int j = lane; j < group; j += 64) {
        const float r = rintf(__fdiv_rn(w[base + j], s));  // round half to even (torch.round)
        q[base + j] = (int8_t)(int)fminf(fmaxf(r, -127.0f), 127.0f);
    }
}

// unpack_int8_weight (nanokv_codec_kernels.py:64-82), _operator_linear
// (MG:145-152): out = bf16(q * scale); the product of an 8-bit integer and a
// bf16 scale is exact in fp32, so out is rounded once.  Eight weights per
// thread when the row length allows 8-byte loads.
__global__ void __launch_bounds__(256) int8_dequant_kernel(const int8_t* __restrict__ q,
                                                           const uint16_t* __restrict__ scale,
                                                           int64_t count, int group,
                                                           uint16_t* __restrict__ out) {
    const int64_t i0 = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 8;
    if (i0 >= count) return;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int64_t i = i0 + e;
        if (i < count)
            out[i] = f32_to_bf16_bits((float)q[i] * bf16_bits_to_f32(scale[i / group]));
    }
}

}  // namespace nkv

extern "C" int nkv_quant_pack(void* stream, const float* coeff, int64_t rows, int r, int group,
                              int scale_dtype, int quant_mode, uint8_t* packed,
                              uint16_t* scales) {
    clear_error();
    NKV_REQUIRE(rows >= 0, NKV_ERR_INVALID, "rows must be >= 0");
    NKV_REQUIRE(r > 0 && r % 8 == 0, NKV_ERR_INVALID, "r must be a positive multiple of 8");
    NKV_REQUIRE(group > 0 && r % group == 0 && group % 8 == 0, NKV_ERR_INVALID,
                "group must divide r and be a multiple of 8");
    NKV_REQUIRE(scale_dtype == NKV_DTYPE_BF16 || scale_dtype == NKV_DTYPE_FP16,
                NKV_ERR_INVALID, "bad scale_dtype");
    NKV_REQUIRE(quant_mode == NKV_QUANT_FP32 || quant_mode == NKV_QUANT_BF16, NKV_ERR_INVALID,
                "bad quant_mode");
    if (rows == 0) return NKV_OK;
    NKV_REQUIRE(coeff && packed && scales, NKV_ERR_INVALID, "null pointer");
    const int64_t threads = rows * (r / group) * quant_lanes(group);
    dim3 grid((unsigned)cdiv(threads, 256));
    hipStream_t s = (hipStream_t)stream;
    if (quant_mode == NKV_QUANT_BF16)
        quant_pack_kernel<NKV_QUANT_BF16><<<grid, 256, 0, s>>>(coeff, rows, r, group, scale_dtype,
                                                                packed, scales);
    else
        quant_pack_kernel<NKV_QUANT_FP32><<<grid, 256, 0, s>>>(coeff, rows, r, group, scale_dtype,
                                                                packed, scales);
    NKV_LAUNCH_CHECK();
    return NKV_OK;
}

extern "C" int nkv_int8_pack(void* stream, const float* w, int64_t rows, int cols, int group,
                             int8_t* q, uint16_t* scale) {
    clear_error();
    NKV_REQUIRE(rows >= 0 && cols > 0, NKV_ERR_INVALID, "bad weight shape");
    NKV_REQUIRE(group > 0 && cols % group == 0, NKV_ERR_INVALID, "group must divide cols");
    if (rows == 0) return NKV_OK;
    NKV_REQUIRE(w && q && scale, NKV_ERR_INVALID, "null pointer");
    const int64_t waves = rows * (cols / group);
    nkv::int8_pack_kernel<<<dim3((unsigned)cdiv(waves, 4)), 256, 0, (hipStream_t)stream>>>(
        w, rows, cols, group, q, scale);
    NKV_LAUNCH_CHECK();
    return NKV_OK;
}

extern "C" int nkv_int8_dequant(void* stream, const int8_t* q, const uint16_t* scale, int64_t rows,
                                int cols, int group, uint16_t* out) {
    clear_error();
    NKV_REQUIRE(rows >= 0 && cols > 0, NKV_ERR_INVALID, "bad weight shape");
    NKV_REQUIRE(group > 0 && cols % group == 0, NKV_ERR_INVALID, "group must divide cols");
    if (rows == 0) return NKV_OK;
    NKV_REQUIRE(q && scale && out, NKV_ERR_INVALID, "null pointer");
    const int64_t count = rows * cols;
    nkv::int8_dequant_kernel<<<dim3((unsigned)cdiv(cdiv(count, 8), 256)), 256, 0,
                               (hipStream_t)stream>>>(q, scale, count, group, out);
    NKV_LAUNCH_CHECK();
    return NKV_OK;
}

extern "C" int nkv_unpack(void* stream, const uint8_t* packed, const uint16_t* scales,
                          int scale_dtype, const int32_t* row_index, int64_t rows, int r,
                          int group, uint16_t* latent) {
    clear_error();
    NKV_REQUIRE(rows >= 0, NKV_ERR_INVALID, "rows must be >= 0");
    NKV_REQUIRE(r > 0 && r % 8 == 0, NKV_ERR_INVALID, "r must be a positive multiple of 8");
    NKV_REQUIRE(group > 0 && r % group == 0 && group % 8 == 0, NKV_ERR_INVALID,
                "group must divide r and be a multiple of 8");
    NKV_REQUIRE(scale_dtype == NKV_DTYPE_BF16 || scale_dtype == NKV_DTYPE_FP16,
                NKV_ERR_INVALID, "bad scale_dtype");
    if (rows == 0) return NKV_OK;
    NKV_REQUIRE(packed && scales && latent, NKV_ERR_INVALID, "null pointer");
    const int64_t threads = rows * (r / 8);
    unpack_kernel<<<dim3((unsigned)cdiv(threads, 256)), 256, 0, (hipStream_t)stream>>>(
        packed, scales, scale_dtype, row_index, rows, r, group, latent);
    NKV_LAUNCH_CHECK();
    return NKV_OK;
}

namespace nkv {

// ------------------------------------------------------------ C64 fit
// The per-chunk joint-head center fit of semantic_residual (MG:301-330):
// centers start as the rows init_rows (the caller's seeded permutation),
// then each round labels every row with its nearest center (the exact fp64
// search, first index on ties) and moves every center that has rows to their
// mean.  The mean is deterministic: the rows of each cluster are listed in
// row order (a stable counting sort), summed in fp64 in that order, rounded
// to fp32 and divided by the count in fp32.

constexpr int FIT_MAXC = 256;

// The initial center rows: in device memory (dev), or a host list carried in
// the kernel arguments (no copy to the device, which would wait for the stream).
struct FitInit {
    const int32_t* dev;
    int32_t v[FIT_MAXC];
    __device__ __forceinline__ int64_t row(int c, int64_t S) const {
        return min(max((int64_t)(dev ? dev[c] : v[c]), (int64_t)0), S - 1);
    }
};

__global__ void __launch_bounds__(256) c64_init_kernel(const float* __restrict__ x, int B, int64_t S,
                                                       int HD, int C,
                                                       FitInit init,
                                                       float* __restrict__ centers) {
    const int64_t total = (int64_t)B * C * HD;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int d = (int)(i % HD);
        const int c = (int)((i / HD) % C);
        const int64_t b = i / ((int64_t)HD * C);
        const int64_t row = init.row(c, S);
        centers[i] = x[(b * S + row) * HD + d];
    }
}

// Eight consecutive values of a row as exact doubles: fp32 or bf16 storage.
template <bool XB>
struct Row8 {
    u32x4 w[XB ? 1 : 2];
    __device__ __forceinline__ void load(const void* base, int64_t at) {
        if constexpr (XB) {
            w[0] = ldg(reinterpret_cast<const u32x4*>(reinterpret_cast<const uint16_t*>(base) + at));
        } else {
            const float* p = reinterpret_cast<const float*>(base) + at;
            w[0] = ldg(reinterpret_cast<const u32x4*>(p));
            w[1] = ldg(reinterpret_cast<const u32x4*>(p + 4));
        }
    }
    __device__ __forceinline__ double get(int e) const {
        if constexpr (XB)
            return (double)__uint_as_float((e & 1) ? (w[0][e >> 1] & 0xffff0000u) : (w[0][e >> 1] << 16));
        else
            return (double)__uint_as_float(w[e >> 2][e & 3]);
    }
};

// The fit's nearest-center search on fp64 MFMA: every product is exact, so
// the decision is that of assign_kernel.  A block of eight waves owns 16 rows
// x 32 centers (two 16 x 16 tiles per wave) and splits HD over its waves
// (wave w: the 32-wide steps w, w + 8, ..); the partial sums meet in LDS and
// are added in wave order.  At C = 64 a chunk of 1,560 rows is 196 blocks of
// eight waves: one wave per 16 rows x 64 centers (the whole HD each, 98 waves
// with work) took 132 us per round, this 22 us.  In a step lane l holds
// row / center l % 16, k 8 (l / 16) .. +8: whole 128-byte lines per row, and
// any order of k is valid for the products.  Bound by latency: each wave's chain
// of loads and dependent products (0.61 GFLOP per round of 64 centers would be 8
// us at the fp64 matrix rate, 32 flop per cycle and SIMD).
// part_d / part_c [center blocks][B * S]: the best center of each block.
// FIRST: the centers are the initial rows of x.  HD % 32 == 0, 16-byte rows.
constexpr int FS_ROWS = 16, FS_CENT = 32, FS_WAVES = 8, FS_AHEAD = 2;

template <bool XB, bool FIRST>
__global__ void __launch_bounds__(64 * FS_WAVES) fit_search_kernel(
    const void* __restrict__ x, const float* __restrict__ centers, FitInit init, int64_t S, int HD,
    int C, double* __restrict__ part_d,
    int32_t* __restrict__ part_c) {
    constexpr bool CB = FIRST && XB;   // the centers' storage is bf16
    // partial sums [wave][tile][element][lane], then ||c||^2 [wave][tile][lane]
    __shared__ double red[FS_WAVES][2][5][64];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int g = lane >> 4, col = lane & 15;
    const int64_t row0 = (int64_t)blockIdx.x * FS_ROWS, b = blockIdx.z;
    const int c0 = blockIdx.y * FS_CENT;
    const int64_t xr = (b * S + min(row0 + col, S - 1)) * HD + 8 * g;
    int64_t cr[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int c = min(c0 + 16 * j + col, C - 1);
        int64_t r = b * C + c;
        if constexpr (FIRST) r = b * S + init.row(c, S);
        cr[j] = r * HD + 8 * g;
    }
    const void* cbase = FIRST ? x : (const void*)centers;
    const int NS = HD / 32;
    Row8<XB> xa[FS_AHEAD];
    Row8<CB> ca[FS_AHEAD][2];
    auto issue = [&](int st, int slot) {
        xa[slot].load(x, xr + 32 * st);
#pragma unroll
        for (int j = 0; j < 2; ++j) ca[slot][j].load(cbase, cr[j] + 32 * st);
    };
    f64x4 acc[2] = {};
    double cc[2] = {0.0, 0.0};
#pragma unroll
    for (int i = 0; i < FS_AHEAD; ++i)
        if (wave + FS_WAVES * i < NS) issue(wave + FS_WAVES * i, i);
    for (int st0 = wave; st0 < NS; st0 += FS_WAVES * FS_AHEAD) {
#pragma unroll
        for (int i = 0; i < FS_AHEAD; ++i) {
            const int st = st0 + FS_WAVES * i;
            if (st >= NS) break;
            const Row8<XB> xv = xa[i];
            Row8<CB> cv[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) cv[j] = ca[i][j];
            if (st + FS_WAVES * FS_AHEAD < NS) issue(st + FS_WAVES * FS_AHEAD, i);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const double a = xv.get(e);
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const double q = cv[j].get(e);
                    acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, q, acc[j], 0, 0, 0);
                    cc[j] = fma(q, q, cc[j]);
                }
            }
        }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
        for (int e = 0; e < 4; ++e) red[wave][j][e][lane] = acc[j][e];
        red[wave][j][4][lane] = cc[j];
    }
    __syncthreads();
    // thread t: row t / 32, center t % 32 of the block.  Element e of lane
    // 16 g + col is row 4 e + g, column col; ||c||^2 is over the four g.
    const int row = t >> 5, cl = t & 31, j = cl >> 4, cc16 = cl & 15;
    double dot = 0.0, cn = 0.0;
    for (int w = 0; w < FS_WAVES; ++w) {
        dot += red[w][j][row >> 2][16 * (row & 3) + cc16];
#pragma unroll
        for (int q = 0; q < 4; ++q) cn += red[w][j][4][16 * q + cc16];
    }
    double bd = cn - 2.0 * dot;
    int bc = c0 + cl < C ? c0 + cl : -1;
#pragma unroll
    for (int off = 1; off < 32; off <<= 1) {
        const double od = __shfl_xor(bd, off);
        const int oc = __shfl_xor(bc, off);
        if (better(od, oc, bd, bc)) { bd = od; bc = oc; }
    }
    if (cl == 0 && row0 + row < S) {
        const int64_t at = (int64_t)blockIdx.y * gridDim.z * S + b * S + row0 + row;
        part_d[at] = bd;
        part_c[at] = bc;
    }
}

// Label of row i (of all B S rows) from the best centers of nc center blocks,
// or (part_d null) the labels as they are.
__device__ __forceinline__ int fit_label(const double* part_d, const int32_t* part_c, int nc,
                                         int64_t total, int64_t i) {
    int c = part_c[i];
    if (!part_d) return c;
    double d = part_d[i];
    for (int k = 1; k < nc; ++k) {
        const double od = part_d[k * total + i];
        const int oc = part_c[k * total + i];
        if (better(od, oc, d, c)) { d = od; c = oc; }
    }
    return c;
}

// labels[i] from more than two center blocks (the update reads one or two itself).
__global__ void __launch_bounds__(256) fit_label_kernel(const double* __restrict__ part_d,
                                                        const int32_t* __restrict__ part_c, int nc,
                                                        int64_t total, int32_t* __restrict__ labels) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < total) labels[i] = fit_label(part_d, part_c, nc, total, i);
}

// One block per (256 columns, cluster c, batch item b): the mean of c's rows.
// The block finds the rows itself, in row order: FU_SCAN labels at a time, a
// ballot per 64 and the counts of the (round, wave) pairs before it (a
// separate stable counting sort by one block took 27 us per round).  Each
// thread then sums its column in that order in fp64, FU_FLY loads in flight
// (22-32 us one at a time, now 11.4 us with the scan: 1,560 rows, 64 clusters;
// bound by the latency of the largest cluster's row list).
// FIRST: an empty cluster's center is its initial row (else it stays).
// The blocks of the first columns write their rows' labels (null: they are
// the labels read).
constexpr int FU_SCAN = 2048, FU_FLY = 16;

template <bool XB>
__global__ void __launch_bounds__(256) fit_update_kernel(
    const void* __restrict__ x, int64_t S, int HD, int C, const double* __restrict__ part_d,
    const int32_t* __restrict__ part_c, int nc, FitInit init, int first,
    float* __restrict__ centers, uint16_t* __restrict__ centers_bf16,
    int32_t* __restrict__ labels, uint8_t* __restrict__ ids) {
    __shared__ int32_t list[FU_SCAN];
    __shared__ int cnt[FU_SCAN / 256][4];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int d = blockIdx.x * 256 + t, c = blockIdx.y;
    const int64_t b = blockIdx.z, total = (int64_t)gridDim.z * S;
    using Raw = typename std::conditional<XB, uint16_t, float>::type;
    const Raw* col = reinterpret_cast<const Raw*>(x) + b * S * HD + d;
    auto at = [&](int64_t row) -> Raw { return ldg(col + row * HD); };
    auto val = [](Raw v) -> float {
        if constexpr (XB) return bf16_bits_to_f32(v);
        else return v;
    };
    double sum = 0.0;
    int64_t n = 0;
    for (int64_t s0 = 0; s0 < S; s0 += FU_SCAN) {
        bool mine[FU_SCAN / 256];
        int before[FU_SCAN / 256];
#pragma unroll
        for (int k = 0; k < FU_SCAN / 256; ++k) {
            const int64_t row = s0 + 256 * k + t;
            // labels outside the table count as its nearest entry
            mine[k] = row < S && min(max(fit_label(part_d, part_c, nc, total, b * S + row), 0), C - 1) == c;
            const uint64_t m = __ballot(mine[k]);
            before[k] = __popcll(m & ((1ull << lane) - 1));
            if (lane == 0) cnt[k][wave] = __popcll(m);
        }
        __syncthreads();
        int run = 0;
#pragma unroll
        for (int k = 0; k < FU_SCAN / 256; ++k) {
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                if (w == wave && mine[k]) list[run + before[k]] = (int32_t)(s0 + 256 * k + t);
                run += cnt[k][w];
            }
        }
        __syncthreads();
        if (blockIdx.x == 0) {
            for (int k = t; k < run; k += 256) {
                if (labels) labels[b * S + list[k]] = c;
                if (ids) ids[b * S + list[k]] = (uint8_t)c;
            }
        }
        if (d < HD) {
            int k = 0;
            for (; k + FU_FLY <= run; k += FU_FLY) {
                Raw v[FU_FLY];
#pragma unroll
                for (int u = 0; u < FU_FLY; ++u) v[u] = at(list[k + u]);
#pragma unroll
                for (int u = 0; u < FU_FLY; ++u) sum += (double)val(v[u]);
            }
            // the rest (fewer than FU_FLY rows) in one flight too; repeats of
            // the last row are not added
            if (k < run) {
                Raw v[FU_FLY];
#pragma unroll
                for (int u = 0; u < FU_FLY; ++u) v[u] = at(list[min(k + u, run - 1)]);
#pragma unroll
                for (int u = 0; u < FU_FLY; ++u)
                    if (k + u < run) sum += (double)val(v[u]);
            }
        }
        n += run;
        __syncthreads();
    }
    if (d >= HD) return;
    const int64_t o = (b * C + c) * HD + d;
    float v;
    if (n > 0) v = __fdiv_rn((float)sum, (float)n);
    else if (first) v = val(at(init.row(c, S)));
    else v = centers[o];
    centers[o] = v;
    if (centers_bf16) centers_bf16[o] = f32_to_bf16_bits(v);
}

__global__ void zero_i32_kernel(int32_t* p, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        p[i] = 0;
}

}  // namespace nkv

// Nearest fp32 center of every row (int32 labels): the fp64 MFMA search, or
// the fp64 VALU search for unaligned operands.
static int launch_assign_f32(hipStream_t s, const float* x, const float* centers, int64_t rows,
                             int C, int HD, int32_t* ids) {
    if (rows <= 0) return NKV_OK;
    if (HD % 16 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0 &&
        reinterpret_cast<uintptr_t>(centers) % 16 == 0) {
        assign_mfma_kernel<4, float><<<dim3((unsigned)cdiv(rows, AM_ROWS)), 256, 0, s>>>(
            x, centers, rows, C, HD, ids);
    } else {
        assign_kernel<4, float><<<dim3((unsigned)cdiv(rows, AS_ROWS)), 256, 0, s>>>(
            x, centers, rows, C, HD, ids);
    }
    NKV_LAUNCH_CHECK();
    return NKV_OK;
}

// The exact bf16-MFMA nearest-center search over every problem of a batch
// (C <= AB_MAXC, HD % AB_SEG == 0, HD <= AB_MAXK, 16-byte aligned rows).
static int launch_assign_batch(hipStream_t s, EncBatch B, bool xb) {
    int64_t rows = 0;
    for (int i = 0; i < B.n; ++i) rows = std::max(rows, B.p[i].M);
    if (rows <= 0) return NKV_OK;
    B.row_blocks = cdiv(rows, AB_ROWS);
    const dim3 grid((unsigned)cdiv(rows, AB_ROWS), (unsigned)B.n);
    const unsigned threads = 64 * AB_WAVES;
    if (xb) {
        const auto kernel = B.id_bytes == 1 ? assign_dma_kernel<1>
                            : B.id_bytes == 2 ? assign_dma_kernel<2> : assign_dma_kernel<4>;
        const int rc = set_smem(kernel, AD_SMEM);
        if (rc) return rc;
        kernel<<<xcd_grid(B.n * B.row_blocks), threads, AD_SMEM, s>>>(B);
    } else {
        if (B.id_bytes == 1) assign_bf16_kernel<1, false><<<grid, threads, 0, s>>>(B);
        else if (B.id_bytes == 2) assign_bf16_kernel<2, false><<<grid, threads, 0, s>>>(B);
        else assign_bf16_kernel<4, false><<<grid, threads, 0, s>>>(B);
    }
    NKV_LAUNCH_CHECK();
    return NKV_OK;
}

static int launch_assign(hipStream_t s, const float* x, const uint16_t* centers, int64_t rows,
                         int C, int HD, void* ids, int id_bytes) {
    if (rows <= 0) return NKV_OK;
    if (C <= AB_MAXC && HD > 0 && HD % AB_SEG == 0 && HD <= AB_MAXK && reinterpret_cast<uintptr_t>(x) % 16 == 0 &&
        reinterpret_cast<uintptr_t>(centers) % 16 == 0) {
        EncBatch B{};
        B.n = 1;
        B.K = HD;
        B.num_centers = C;
        B.id_bytes = id_bytes;
        B.p[0].x = x;
        B.p[0].ldx = HD;
        B.p[0].centers = centers;
        B.p[0].ids = ids;
        B.p[0].M = rows;
        return launch_assign_batch(s, B, false);
    }
    if (HD > 0 && HD % 16 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0 &&
        reinterpret_cast<uintptr_t>(centers) % 8 == 0) {
        dim3 grid((unsigned)cdiv(rows, AM_ROWS));
        if (id_bytes == 1)
            assign_mfma_kernel<1><<<grid, 256, 0, s>>>(x, centers, rows, C, HD, ids);
        else if (id_bytes == 2)
            assign_mfma_kernel<2><<<grid, 256, 0, s>>>(x, centers, rows, C, HD, ids);
        else
            assign_mfma_kernel<4><<<grid, 256, 0, s>>>(x, centers, rows, C, HD, ids);
        NKV_LAUNCH_CHECK();
        return NKV_OK;
    }
    dim3 grid((unsigned)cdiv(rows, AS_ROWS));
    if (id_bytes == 1)
        assign_kernel<1><<<grid, 256, 0, s>>>(x, centers, rows, C, HD, ids);
    else if (id_bytes == 2)
        assign_kernel<2><<<grid, 256, 0, s>>>(x, centers, rows, C, HD, ids);
    else
        assign_kernel<4><<<grid, 256, 0, s>>>(x, centers, rows, C, HD, ids);
    NKV_LAUNCH_CHECK();
    return NKV_OK;
}

static int check_ids(int C, int id_bytes) {
    NKV_REQUIRE(id_bytes == 1 || id_bytes == 2 || id_bytes == 4, NKV_ERR_INVALID,
                "id_bytes must be 1, 2 or 4");
    NKV_REQUIRE(C > 0, NKV_ERR_INVALID, "need at least one center");
    NKV_REQUIRE(!(id_bytes == 1 && C > 256), NKV_ERR_INVALID, "uint8 ids need C <= 256");
    NKV_REQUIRE(!(id_bytes == 2 && C > 65536), NKV_ERR_INVALID, "uint16 ids need C <= 65536");
    return NKV_OK;
}

namespace {
size_t fit_ws_align(size_t n) { return (n + 255) / 256 * 256; }
}  // namespace

// Workspace of a fit: the best distance and center of every row per block of
// FS_CENT centers.
static size_t fit_part_bytes(int B, int64_t S, int C, size_t elem) {
    return fit_ws_align((size_t)cdiv(C, FS_CENT) * B * S * elem);
}

// What the search by whole rows needs.
static size_t fit_label_bytes(int B, int64_t S) { return fit_ws_align((size_t)B * S * sizeof(int32_t)); }

extern "C" size_t nkv_c64_fit_workspace_size(int B, int64_t S, int C) {
    if (B <= 0 || S <= 0 || C <= 0) return 0;
    return fit_part_bytes(B, S, C, sizeof(double)) + fit_part_bytes(B, S, C, sizeof(int32_t));
}

extern "C" int nkv_c64_fit(void* stream, const float* x, int B, int64_t S, int HD, int C,
                           int iterations, const int32_t* init_rows, float* centers,
                           int32_t* labels, void* workspace, size_t workspace_bytes) {
    nkv_c64_fit_args a{};
    a.x = x;
    a.B = B;
    a.S = S;
    a.HD = HD;
    a.C = C;
    a.iterations = iterations;
    a.init_rows = init_rows;
    a.centers = centers;
    a.labels = labels;
    a.workspace = workspace;
    a.workspace_bytes = workspace_bytes;
    return nkv_c64_fit_rows(stream, &a);
}

extern "C" int nkv_c64_fit_rows(void* stream, const nkv_c64_fit_args* a) {
    clear_error();
    NKV_REQUIRE(a, NKV_ERR_INVALID, "null args");
    const int B = a->B, HD = a->HD, C = a->C;
    const int64_t S = a->S;
    NKV_REQUIRE(B >= 0 && S >= 0 && HD > 0, NKV_ERR_INVALID, "bad shape");
    NKV_REQUIRE(a->iterations >= 0, NKV_ERR_INVALID, "iterations must be >= 0");
    if (B == 0 || S == 0) return NKV_OK;
    NKV_REQUIRE(C >= 1 && C <= S && C <= FIT_MAXC, NKV_ERR_INVALID,
                "C64 clusters must be in [1, min(S, 256)]");
    NKV_REQUIRE(S < INT32_MAX, NKV_ERR_INVALID, "rows must fit in 32 bits");
    NKV_REQUIRE((a->x || a->x_bf16) && (a->init_rows || a->init_rows_host) && a->centers && a->labels,
                NKV_ERR_INVALID, "null pointer");
    NKV_REQUIRE(!(a->x && a->x_bf16), NKV_ERR_INVALID, "give x or x_bf16, not both");
    const bool xb = a->x_bf16 != nullptr;
    const void* x = xb ? (const void*)a->x_bf16 : (const void*)a->x;
    // the fp64 MFMA search: whole 32-wide steps, 16-byte rows; a workspace too
    // small for its partial results takes the search by whole rows, which keeps
    // their labels alone (fp32 rows)
    const bool fits = a->workspace_bytes >= nkv_c64_fit_workspace_size(B, S, C);
    const bool steps = HD % 32 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0 &&
                       reinterpret_cast<uintptr_t>(a->centers) % 16 == 0 && B <= 65535 &&
                       reinterpret_cast<uintptr_t>(a->workspace) % 8 == 0;
    const bool mfma = steps && fits, rounds = a->iterations > 0;
    NKV_REQUIRE(a->workspace && (fits || (!xb && a->workspace_bytes >= fit_label_bytes(B, S))),
                NKV_ERR_WORKSPACE, "workspace missing or smaller than nkv_c64_fit_workspace_size()");
    NKV_REQUIRE(!xb || (steps && rounds), NKV_ERR_UNSUPPORTED,
                "a bf16 fit needs HD % 32 == 0, 16-byte aligned rows and at least one round");
    NKV_REQUIRE(rounds || !(a->centers_bf16 || a->ids_u8), NKV_ERR_UNSUPPORTED,
                "bf16 centers and uint8 ids need at least one round");
    unsigned char* ws = reinterpret_cast<unsigned char*>(a->workspace);
    double* part_d = reinterpret_cast<double*>(ws);
    int32_t* part_c = reinterpret_cast<int32_t*>(ws + (mfma ? fit_part_bytes(B, S, C, sizeof(double)) : 0));
    FitInit init{};
    init.dev = a->init_rows;
    if (!init.dev) std::copy(a->init_rows_host, a->init_rows_host + C, init.v);
    hipStream_t s = (hipStream_t)stream;
    if (!mfma || !rounds) {
        const int64_t elems = (int64_t)B * C * HD;
        c64_init_kernel<<<dim3((unsigned)std::min<int64_t>(cdiv(elems, 256), 4096)), 256, 0, s>>>(
            a->x, B, S, HD, C, init, a->centers);
        NKV_LAUNCH_CHECK();
    }
    if (!rounds) {
        // no round: the labels stay zero, as the reference initialises them
        zero_i32_kernel<<<dim3((unsigned)std::min<int64_t>(cdiv((int64_t)B * S, 256), 4096)), 256,
                          0, s>>>(a->labels, (int64_t)B * S);
        NKV_LAUNCH_CHECK();
        return NKV_OK;
    }
    const int64_t total = (int64_t)B * S;
    const int ncb = (int)cdiv(C, FS_CENT);
    for (int it = 0; it < a->iterations; ++it) {
        const bool first = mfma && it == 0, last = it + 1 == a->iterations;
        const double* pd = part_d;
        const int32_t* pc = part_c;
        int nc = ncb;
        if (mfma) {
            const dim3 grid((unsigned)cdiv(S, FS_ROWS), (unsigned)ncb, (unsigned)B);
            auto run = [&](auto kernel) {
                kernel<<<grid, 64 * FS_WAVES, 0, s>>>(x, a->centers, init, S, HD, C, part_d, part_c);
            };
            if (xb) first ? run(fit_search_kernel<true, true>) : run(fit_search_kernel<true, false>);
            else first ? run(fit_search_kernel<false, true>) : run(fit_search_kernel<false, false>);
            NKV_LAUNCH_CHECK();
            if (ncb > 2) {
                fit_label_kernel<<<dim3((unsigned)cdiv(total, 256)), 256, 0, s>>>(part_d, part_c, ncb,
                                                                                  total, a->labels);
                NKV_LAUNCH_CHECK();
                pd = nullptr;
                pc = a->labels;
            }
        } else {
            for (int b = 0; b < B; ++b) {
                const int rc = launch_assign_f32(s, a->x + b * S * HD, a->centers + (int64_t)b * C * HD,
                                                 S, C, HD, part_c + b * S);
                if (rc) return rc;
            }
            pd = nullptr;
        }
        const dim3 grid((unsigned)cdiv(HD, 256), (unsigned)C, (unsigned)B);
        auto run = [&](auto kernel) {
            kernel<<<grid, 256, 0, s>>>(x, S, HD, C, pd, pc, nc, init, first ? 1 : 0,
                                        a->centers, last ? a->centers_bf16 : nullptr,
                                        pc == a->labels ? nullptr : a->labels,
                                        last ? a->ids_u8 : nullptr);
        };
        if (xb) run(fit_update_kernel<true>);
        else run(fit_update_kernel<false>);
        NKV_LAUNCH_CHECK();
    }
    return NKV_OK;
}

extern "C" int nkv_assign(void* stream, const float* x, const uint16_t* centers, int64_t rows,
                          int C, int HD, void* ids, int id_bytes) {
    clear_error();
    NKV_REQUIRE(rows >= 0 && HD > 0, NKV_ERR_INVALID, "rows must be >= 0 and HD > 0");
    int rc = check_ids(C, id_bytes);
    if (rc) return rc;
    if (rows == 0) return NKV_OK;
    NKV_REQUIRE(x && centers && ids, NKV_ERR_INVALID, "null pointer");
    return launch_assign((hipStream_t)stream, x, centers, rows, C, HD, ids, id_bytes);
}

namespace {

// Checks of one encode problem; the batch's shape and settings are those of
// its first problem.
int check_encode(const nkv_encode_args* a, const nkv_encode_args* first) {
    NKV_REQUIRE(a, NKV_ERR_INVALID, "null args");
    NKV_REQUIRE(a->rows >= 0, NKV_ERR_INVALID, "rows must be >= 0");
    NKV_REQUIRE(a->HD > 0 && a->HD % 32 == 0, NKV_ERR_INVALID, "HD must be a multiple of 32");
    int rc = check_codec_layout(a->r, a->group, a->scale_dtype);
    if (rc) return rc;
    NKV_REQUIRE(a->quant_mode == NKV_QUANT_FP32 || a->quant_mode == NKV_QUANT_BF16,
                NKV_ERR_INVALID, "bad quant_mode");
    if (a->centers) {
        rc = check_ids(a->num_centers, a->id_bytes);
        if (rc) return rc;
        NKV_REQUIRE(a->ids, NKV_ERR_INVALID, "ids required with centers");
    }
    NKV_REQUIRE(!(a->x && a->x_bf16), NKV_ERR_INVALID, "give x or x_bf16, not both");
    NKV_REQUIRE(a->x_stride == 0 || a->x_stride >= a->HD, NKV_ERR_INVALID,
                "x_stride must be 0 or at least HD");
    if (first != a) {
        NKV_REQUIRE(a->HD == first->HD && a->r == first->r && a->group == first->group &&
                        a->scale_dtype == first->scale_dtype &&
                        a->quant_mode == first->quant_mode &&
                        (a->centers != nullptr) == (first->centers != nullptr) &&
                        a->num_centers == first->num_centers && a->id_bytes == first->id_bytes &&
                        a->ids_in == first->ids_in &&
                        (a->x_bf16 != nullptr) == (first->x_bf16 != nullptr) &&
                        (a->mean != nullptr) == (first->mean != nullptr),
                    NKV_ERR_INVALID,
                    "the problems of one encode batch must share HD, r, group, scale and quant "
                    "settings, center count and id type, and the input dtype");
    }
    if (a->rows == 0) return NKV_OK;
    NKV_REQUIRE((a->x || a->x_bf16) && a->w_enc && a->coeff && a->packed && a->scales,
                NKV_ERR_INVALID, "null pointer");
    return NKV_OK;
}

// How an encode with a workspace runs: rows per pass (0: not at all) and
// problem, splits of the search, workspace bytes.
struct EncPlan {
    int64_t pass;
    int splits, cols;        // columns of a projection tile
    size_t dots, cnorm, planes, resid, bytes;   // per problem, bytes in all
};

// At most ENC_PASS rows of all problems in one pass, so that the workspace
// does not grow with the input; 4,096 rows are 32 row tiles of the search and
// 64 x 6 tiles of the projection at r = 384: more fill the chip no better.
constexpr int64_t ENC_PASS = 4096;

// Whether the GEMMs over the workspace beat the kernels without one.  us
// without / with a workspace, in a graph, r = 64 unless stated.
//
// The batched kernels (HD % 256 == 0, to search at most 256 centers) read every
// row once; their time is flat until blocks of 32 rows x 192 columns fill the chip:
//   one pass, no search, 780 rows: HD 512 12 / 11, 1,024 16 / 13, 3,072 33 / 24; a
//   call from the host costs 4 us more with one (the scratch, a launch more): 13 /
//   17 and 17 / 17 at 512 and 1,024.
//   one pass, a search of 16 centers, 1,560 rows: HD 256 bf16 22 / 20, fp32 24 / 26
//   (300 rows 24 / 24); 512 bf16 28 / 25, fp32 29 / 28; two problems of 512 and 64
//   centers 28 / 27, from the host 31.6 / 33.5.
//   6,000 rows, two passes, 64 centers: HD 512 r = 384 43 / 57, 3,072 79 / 93, r = 384
//   120 / 103 (two column blocks of the projection); fp32 rows, which a search
//   splits in two planes, 135 / 142.
//
// The general kernels (other widths; more centers) search in fp64, 64 centers at
// least, and project 64 x 64 tiles:
//   no search: HD 128 9 / 9, 384 12 / 10 (1,560 rows); 12,480 rows 14 / 45 at 384, 35 /
//   72 at 1,152 (r = 384 67 / 81); 6,000 rows of 3,200 77 / 60, r = 384 88 / 69.
//   1,560 rows, centers x HD: 64 x 128 21 / 22, 64 x 384 37 / 30, 300 x 128 30 / 24.
//   12,480 rows: 64 x 384 103 / 144, 300 x 128 83 / 115, 64 x 640 153 / 152, 1,024 x 128
//   148 / 146, 300 x 384 178 / 152.
bool enc_gemm_pays(const nkv_encode_args* a, int n, bool search, int64_t rows, int64_t pass) {
    const bool one_pass = rows <= pass;
    if (a->HD % 256 || (search && a->num_centers > AB_MAXC)) {
        if (search)
            return (int64_t)std::max(a->num_centers, 64) * a->HD >= (one_pass ? 24576 : 40960);
        return one_pass ? a->HD >= 384 : a->HD >= 2048 && (a->r > EP_COLS || rows <= 2 * pass);
    }
    if (!one_pass) return a->HD >= 2048 && a->r > EP_COLS && (!search || a->x_bf16);
    if (!search || n > 1) return a->HD >= 1024;
    return a->x_bf16 || a->HD >= 512 || rows <= 512;
}

EncPlan enc_plan(const nkv_encode_args* a, int n) {
    EncPlan p{};
    const bool search = a->centers && !a->ids_in;
    int64_t rows = 0;
    for (int i = 0; i < n; ++i) rows = std::max(rows, a[i].rows);
    // whole stages; a decision keeps its row's centers in registers,
    // its bound holds to SD_MAXK; byte offsets of rows in 32 bits
    if (rows == 0 || a->HD % 128 || (search && (a->num_centers > SD_MAXC || a->HD > SD_MAXK))) return p;
    if ((int64_t)std::max(a->r, search ? a->num_centers : 0) * a->HD * 2 > UINT32_MAX) return p;
    for (int i = 0; i < n; ++i)
        if (a[i].x_stride > (1 << 20)) return p;
    const int64_t pass = std::max<int64_t>(ENC_PASS / n / DotsTile::TM, 1) * DotsTile::TM;
    if (!enc_gemm_pays(a, n, search, rows, pass)) return p;
    p.pass = std::min(rows, pass);
    auto up = [](size_t b) { return (b + 255) / 256 * 256; };
    p.resid = up((size_t)p.pass * a->HD * 2);
    // the narrowest tile whose blocks run in one round of the 256 CUs (one
    // block each: three stages of 128 k take 96 or 120 KB of LDS), else the
    // widest (72 KB, two blocks per CU)
    const int64_t row_tiles = n * cdiv(p.pass, Proj64::TM);
    p.cols = row_tiles * cdiv(a->r, 64) <= 256 ? 64 : row_tiles * cdiv(a->r, 96) <= 256 ? 96 : 128;
    if (search) {
        const int64_t tiles = n * cdiv(p.pass, DotsTile::TM) * cdiv(a->num_centers, DotsTile::TN);
        const int stages = (a->x_bf16 ? 1 : 2) * (a->HD / 64);
        // one block per CU (128 KB of LDS): splits up to a full chip, of at
        // least eight stages each
        p.splits = (int)std::max<int64_t>(1, std::min<int64_t>({256 / tiles, stages / 8, 16}));
        p.dots = up((size_t)p.splits * p.pass * ((a->num_centers + 3) & ~3) * 4);
        p.cnorm = up((size_t)p.splits * a->num_centers * 4);
        if (!a->x_bf16) p.planes = 2 * up((size_t)p.pass * a->HD * 2);
    }
    p.bytes = n * (p.resid + p.dots + p.cnorm + p.planes);
    return p;
}

int encode_staged(hipStream_t s, const EncBatch& B, bool xb, bool search, const nkv_encode_args* a,
                  const EncPlan& pl) {
    EncWsBatch W{};
    W.e = B;
    W.splits = pl.splits;
    const int n = B.n;
    int64_t rows = 0;
    unsigned char* ws = reinterpret_cast<unsigned char*>(a->workspace);
    for (int i = 0; i < n; ++i) {
        rows = std::max(rows, B.p[i].M);
        EncWs& w = W.w[i];
        auto take = [&](size_t b) { unsigned char* p = ws; ws += b; return p; };
        w.resid = reinterpret_cast<uint16_t*>(take(pl.resid));
        w.dots = reinterpret_cast<float*>(take(pl.dots));
        w.cnorm = reinterpret_cast<float*>(take(pl.cnorm));
        unsigned char* planes = take(pl.planes);
        w.ld = xb ? B.p[i].ldx : B.K;
        w.xh = reinterpret_cast<const uint16_t*>(planes);
        w.xl = xb ? nullptr : reinterpret_cast<const uint16_t*>(planes + pl.planes / 2);
    }
    W.e.scale_dtype = a->scale_dtype;
    W.e.quant_mode = a->quant_mode;
    for (int64_t m0 = 0; m0 < rows; m0 += pl.pass) {
        W.m0 = m0;
        W.rows = (int)std::min(pl.pass, rows - m0);
        if (xb)
            for (int i = 0; i < n; ++i) W.w[i].xh = B.p[i].xb + m0 * B.p[i].ldx;
        if (search) {
            if (!xb) {
                const int64_t units = (int64_t)W.rows * (B.K / 8);
                split_rows_kernel<<<dim3((unsigned)std::min<int64_t>(cdiv(units, 256), 4096), n), 256, 0, s>>>(W);
                NKV_LAUNCH_CHECK();
            }
            const unsigned tiles = (unsigned)(cdiv(W.rows, DotsTile::TM) * cdiv(B.num_centers, DotsTile::TN));
            const int rc = set_smem(search_dots_kernel, DotsTile::SMEM);
            if (rc) return rc;
            search_dots_kernel<<<dim3(tiles, pl.splits, n), DotsTile::THREADS, DotsTile::SMEM, s>>>(W);
            NKV_LAUNCH_CHECK();
        }
        const dim3 dgrid((unsigned)cdiv(W.rows, 4), n);
        auto decide = [&](auto k) { k<<<dgrid, 256, 0, s>>>(W); };
        if (!search) {
            xb ? decide(decide_kernel<1, true, false>) : decide(decide_kernel<1, false, false>);
        } else if (B.id_bytes == 1) {
            xb ? decide(decide_kernel<1, true, true>) : decide(decide_kernel<1, false, true>);
        } else if (B.id_bytes == 2) {
            xb ? decide(decide_kernel<2, true, true>) : decide(decide_kernel<2, false, true>);
        } else {
            xb ? decide(decide_kernel<4, true, true>) : decide(decide_kernel<4, false, true>);
        }
        NKV_LAUNCH_CHECK();
        auto project = [&](auto tile, auto kernel) -> int {
            using T = decltype(tile);
            W.e.qgroup = T::TN % a->group == 0 ? a->group : 0;
            const int rc = set_smem(kernel, T::SMEM);
            if (rc) return rc;
            kernel<<<xcd_grid(n * cdiv(W.rows, T::TM) * cdiv(B.r, T::TN)), T::THREADS, T::SMEM, s>>>(W);
            NKV_LAUNCH_CHECK();
            return NKV_OK;
        };
        const int rc = pl.cols == 64   ? project(Proj64{}, project_kernel<Proj64>)
                       : pl.cols == 96 ? project(Proj96{}, project_kernel<Proj96>)
                                       : project(Proj128{}, project_kernel<Proj128>);
        if (rc) return rc;
    }
    if (W.e.qgroup) return NKV_OK;
    const dim3 qgrid((unsigned)cdiv(rows * (B.r / a->group) * quant_lanes(a->group), 256), (unsigned)n);
    if (a->quant_mode == NKV_QUANT_BF16)
        quant_pack_batch_kernel<NKV_QUANT_BF16><<<qgrid, 256, 0, s>>>(B, a->group, a->scale_dtype);
    else
        quant_pack_batch_kernel<NKV_QUANT_FP32><<<qgrid, 256, 0, s>>>(B, a->group, a->scale_dtype);
    NKV_LAUNCH_CHECK();
    return NKV_OK;
}

int encode_batch(hipStream_t s, const nkv_encode_args* a, int n) {
    NKV_REQUIRE(a && n >= 1 && n <= ENC_MAXB, NKV_ERR_INVALID, "1..8 encode problems");
    for (int i = 0; i < n; ++i) {
        int rc = check_encode(a + i, a);
        if (rc) return rc;
    }
    const int HD = a->HD, r = a->r;
    const bool xb = a->x_bf16 != nullptr;
    EncBatch B{};
    B.n = n;
    B.K = HD;
    B.r = r;
    B.num_centers = a->num_centers;
    B.id_bytes = a->id_bytes;
    bool aligned = true;
    int64_t rows = 0;
    for (int i = 0; i < n; ++i) {
        const nkv_encode_args& q = a[i];
        EncProb& P = B.p[i];
        P.x = q.x;
        P.xb = q.x_bf16;
        P.ldx = q.x_stride ? q.x_stride : HD;
        P.centers = q.centers;
        P.ids = q.ids;
        P.mean = q.mean;
        P.w_enc = q.w_enc;
        P.coeff = q.coeff;
        P.packed = q.packed;
        P.scales = q.scales;
        P.M = q.rows;
        rows = std::max(rows, q.rows);
        const uintptr_t xp = reinterpret_cast<uintptr_t>(xb ? (const void*)q.x_bf16 : (const void*)q.x);
        aligned = aligned && xp % 16 == 0 && (P.ldx * (xb ? 2 : 4)) % 16 == 0 &&
                  (!q.centers || reinterpret_cast<uintptr_t>(q.centers) % 16 == 0);
    }
    if (rows == 0) return NKV_OK;
    // the batched kernels: the exact bf16-MFMA search (C <= 256) and the
    // staged projection; a bf16 input takes only those
    const bool fast_search = a->num_centers <= AB_MAXC && HD % AB_SEG == 0 && HD <= AB_MAXK;
    const bool fast_proj = HD % 256 == 0;
    static_assert(256 % EP_KS == 0, "the staged projection needs HD % EP_KS == 0");
    const bool search = a->centers && !a->ids_in;
    NKV_REQUIRE(!xb || (aligned && fast_proj && (!search || fast_search)), NKV_ERR_UNSUPPORTED,
                "a bf16 input needs HD % 256 == 0, 16-byte aligned rows and, to search, at most 256 "
                "centers and HD <= 16384");
    // (a strided fp32 input needs the 16-byte kernels; see the launches below)
    const bool strided_ok = aligned && fast_proj && (!search || fast_search);
    bool packed_rows = true, w16 = reinterpret_cast<uintptr_t>(a->workspace) % 16 == 0;
    for (int i = 0; i < n; ++i) {
        packed_rows = packed_rows && B.p[i].ldx == HD;
        w16 = w16 && reinterpret_cast<uintptr_t>(B.p[i].w_enc) % 16 == 0;
    }
    if (a->workspace && aligned && w16 && (packed_rows || strided_ok)) {
        const EncPlan pl = enc_plan(a, n);
        if (pl.pass > 0 && a->workspace_bytes >= pl.bytes) return encode_staged(s, B, xb, search, a, pl);
    }
    int rc = NKV_OK;
    if (search) {
        if (fast_search && aligned) {
            rc = launch_assign_batch(s, B, xb);
        } else {
            for (int i = 0; i < n && !rc; ++i) {
                NKV_REQUIRE(B.p[i].ldx == HD, NKV_ERR_UNSUPPORTED,
                            "a strided fp32 input needs HD % 256 == 0, at most 256 centers and "
                            "16-byte aligned rows");
                rc = launch_assign(s, B.p[i].x, B.p[i].centers, B.p[i].M, B.num_centers, HD,
                                   B.p[i].ids, B.id_bytes);
            }
        }
        if (rc) return rc;
    }
    if (fast_proj && aligned) {
        B.row_blocks = cdiv(rows, EP_ROWS);
        // groups that do not straddle column blocks are quantised in the same launch
        B.qgroup = EP_COLS % a->group == 0 ? a->group : 0;
        B.scale_dtype = a->scale_dtype;
        B.quant_mode = a->quant_mode;
        const unsigned grid = xcd_grid(n * cdiv(r, EP_COLS) * B.row_blocks);
        const auto kernel = xb ? encode_proj_kernel<true> : encode_proj_kernel<false>;
        const int smem = xb ? EncProjFmt<true>::SMEM : EncProjFmt<false>::SMEM;
        rc = set_smem(kernel, smem);
        if (rc) return rc;
        kernel<<<grid, 64 * EP_WAVES, smem, s>>>(B);
        NKV_LAUNCH_CHECK();
        if (B.qgroup) return NKV_OK;
    } else {
        for (int i = 0; i < n; ++i) {
            if (B.p[i].M == 0) continue;
            NKV_REQUIRE(B.p[i].ldx == HD, NKV_ERR_UNSUPPORTED,
                        "a strided fp32 input needs HD % 256 == 0 and 16-byte aligned rows");
            EncodeA al;
            al.x = B.p[i].x;
            al.centers = B.p[i].centers;
            al.ids = B.p[i].ids;
            al.id_bytes = B.id_bytes;
            al.num_centers = B.num_centers;
            al.mean = B.p[i].mean;
            al.M = B.p[i].M;
            al.K = HD;
            dim3 grid((unsigned)cdiv(al.M, GT_M), (unsigned)cdiv(r, GT_N));
            encode_gemm_kernel<<<grid, 256, 0, s>>>(al, B.p[i].w_enc, r, B.p[i].coeff);
            NKV_LAUNCH_CHECK();
        }
    }
    const dim3 qgrid((unsigned)cdiv(rows * (r / a->group) * quant_lanes(a->group), 256), (unsigned)n);
    if (a->quant_mode == NKV_QUANT_BF16)
        quant_pack_batch_kernel<NKV_QUANT_BF16><<<qgrid, 256, 0, s>>>(B, a->group, a->scale_dtype);
    else
        quant_pack_batch_kernel<NKV_QUANT_FP32><<<qgrid, 256, 0, s>>>(B, a->group, a->scale_dtype);
    NKV_LAUNCH_CHECK();
    return NKV_OK;
}

}  // namespace

extern "C" size_t nkv_encode_workspace_size(const nkv_encode_args* a, int n) {
    clear_error();
    if (!a || n < 1 || n > ENC_MAXB) return 0;
    for (int i = 0; i < n; ++i)
        if (check_encode(a + i, a)) return 0;
    return enc_plan(a, n).bytes;
}

extern "C" int nkv_encode(void* stream, const nkv_encode_args* a) {
    clear_error();
    return encode_batch((hipStream_t)stream, a, 1);
}

extern "C" int nkv_encode_batch(void* stream, const nkv_encode_args* args, int n) {
    clear_error();
    return encode_batch((hipStream_t)stream, args, n);
}

namespace {

int check_decode(const nkv_decode_args* a) {
    NKV_REQUIRE(a, NKV_ERR_INVALID, "null args");
    const nkv_codec& c = a->codec;
    NKV_REQUIRE(a->B >= 1 && a->N >= 0 && a->rows >= 0, NKV_ERR_INVALID, "bad B/N/rows");
    NKV_REQUIRE(a->HD > 0 && a->HD % 32 == 0, NKV_ERR_INVALID, "HD must be a multiple of 32");
    int rc = check_codec_layout(c.r, c.group, c.scale_dtype);
    if (rc) return rc;
    NKV_REQUIRE(a->row_index || a->rows == a->N, NKV_ERR_INVALID,
                "rows must equal N without row_index");
    NKV_REQUIRE(c.n_segments == 0, NKV_ERR_UNSUPPORTED,
                "nkv_decode takes a flat codec; decode segments one at a time");
    if (c.centers) {
        rc = check_ids(c.num_centers, c.id_bytes);
        if (rc) return rc;
        NKV_REQUIRE(c.ids, NKV_ERR_INVALID, "ids required with centers");
    }
    if (a->rows == 0) return NKV_OK;
    NKV_REQUIRE(c.packed && c.scales && c.w_dec && a->out, NKV_ERR_INVALID, "null pointer");
    return NKV_OK;
}

// Batch item b of a decode call as one problem.
DecProb dec_problem(const nkv_decode_args* a, int b) {
    const nkv_codec& c = a->codec;
    DecProb p;
    p.packed = c.packed + (int64_t)b * a->N * (c.r / 2);
    p.scales = c.scales + (int64_t)b * a->N * (c.r / c.group);
    p.ids = c.ids ? (const void*)((const uint8_t*)c.ids + (int64_t)b * a->N * c.id_bytes) : nullptr;
    p.centers = c.centers ? c.centers + (int64_t)b * c.centers_batch_stride : nullptr;
    p.row_index = a->row_index;
    p.out = a->out + (int64_t)b * a->rows * a->HD;
    p.M = a->rows;
    p.id_bytes = c.id_bytes;
    p.num_centers = c.num_centers;
    return p;
}

// The staged kernel's 8- and 16-byte accesses (r % 32 == 0 and HD % 32 == 0
// keep every row aligned when its base is).
bool dec_aligned(const DecProb& p, const uint16_t* w) {
    auto at = [](const void* q, uintptr_t n) { return reinterpret_cast<uintptr_t>(q) % n == 0; };
    return at(p.packed, 8) && at(p.centers, 16) && at(p.out, 16) && at(w, 16);
}

template <int MI, int WR, int WC>
int launch_decode_tiles(hipStream_t s, DecBatch& B, int64_t rows) {
    using F = DecFmt<MI, WR, WC>;
    const int rc = set_smem(decode_tile_kernel<MI, WR, WC>, F::SMEM);
    if (rc) return rc;
    const int64_t items = B.n * cdiv(rows, F::ROWS) * cdiv(B.HD, F::COLS);
    NKV_REQUIRE(items < INT32_MAX - 8, NKV_ERR_UNSUPPORTED, "decode grid too large");
    B.row_blocks = (uint32_t)cdiv(rows, F::ROWS);
    decode_tile_kernel<MI, WR, WC><<<xcd_grid(items), F::THREADS, F::SMEM, s>>>(B);
    NKV_LAUNCH_CHECK();
    return NKV_OK;
}

int launch_decode(hipStream_t s, const nkv_decode_args* first, const DecProb* p, int n) {
    const nkv_codec& c = first->codec;
    for (int i0 = 0; i0 < n; i0 += DEC_MAXB) {
        DecBatch B{};
        B.n = std::min(n - i0, DEC_MAXB);
        B.w = c.w_dec;
        B.mean = c.mean;
        B.HD = first->HD;
        B.r = c.r;
        B.group = c.group;
        B.scale_dtype = c.scale_dtype;
        int64_t rows = 0, big = 0;
        for (int i = 0; i < B.n; ++i) {
            B.p[i] = p[i0 + i];
            rows = std::max(rows, B.p[i].M);
            big += cdiv(B.p[i].M, DecBig::ROWS) * cdiv(B.HD, DecBig::COLS);
        }
        // one round of 128 x 256 tiles over the 256 CUs, or more: those; below,
        // 64 x 128 tiles (four times the blocks).  1,017 x 2,048 at r = 256:
        // 9.4 us with the small tiles on 256 CUs, 64 blocks of the large ones
        const int rc = big >= 256 ? launch_decode_tiles<2, 2, 4>(s, B, rows)
                                  : launch_decode_tiles<1, 2, 2>(s, B, rows);
        if (rc) return rc;
    }
    return NKV_OK;
}

// Few rows of a low rank: decode_gemm_kernel's one tile per block starts sooner
// than the staged tiles' first slice.  us in a graph, that kernel / the staged
// ones: no centers, 1 x 256 2.80 / 3.61 (r = 32), 3.70 / 4.24 (96), 5.85 / 5.97
// (256), 7.64 / 7.55 (384); 300 x 3,072 4.17 / 4.28 (r = 64), 5.10 / 5.05 (128); 600 x
// 3,072 at r = 64 4.73 / 4.60; 24 x 256 at r = 256 6.26 / 6.14.  With centers, which
// it adds two bytes at a time: 2 x 3,072 3.39 / 4.06 (r = 32), 6.47 / 6.48 (256);
// 4 x 3,072 at r = 64 4.27 / 4.18.
bool plain_decode_pays(const nkv_decode_args* a) {
    const nkv_codec& c = a->codec;
    if (a->B != 1 || c.r > 256) return false;
    if (c.centers) return a->rows <= 2;
    return a->rows <= 16 || (c.r <= 96 && a->rows * a->HD <= (1 << 20));
}

int decode_one(hipStream_t s, const nkv_decode_args* a) {
    const nkv_codec& c = a->codec;
    if (a->rows == 0) return NKV_OK;
    bool staged = !plain_decode_pays(a);
    for (int b = 0; b < a->B; ++b) staged = staged && dec_aligned(dec_problem(a, b), c.w_dec);
    if (staged) {
        DecProb p[DEC_MAXB];
        for (int b0 = 0; b0 < a->B; b0 += DEC_MAXB) {
            const int nb = std::min(a->B - b0, DEC_MAXB);
            for (int b = 0; b < nb; ++b) p[b] = dec_problem(a, b0 + b);
            const int rc = launch_decode(s, a, p, nb);
            if (rc) return rc;
        }
        return NKV_OK;
    }
    dim3 grid((unsigned)cdiv(a->rows, GT_M), (unsigned)cdiv(a->HD, GT_N));
    for (int b = 0; b < a->B; ++b) {
        const DecProb p = dec_problem(a, b);
        DecodeA al;
        al.packed = p.packed;
        al.scales = p.scales;
        al.row_index = p.row_index;
        al.scale_dtype = c.scale_dtype;
        al.group = c.group;
        al.M = p.M;
        al.K = c.r;
        DecodeEpi ep;
        ep.centers = p.centers;
        ep.ids = p.ids;
        ep.id_bytes = c.id_bytes;
        ep.num_centers = c.num_centers;
        ep.row_index = p.row_index;
        ep.mean = c.mean;
        decode_gemm_kernel<<<grid, 256, 0, s>>>(al, ep, c.w_dec, a->HD, p.out);
        NKV_LAUNCH_CHECK();
    }
    return NKV_OK;
}

}  // namespace

extern "C" int nkv_decode(void* stream, const nkv_decode_args* a) {
    clear_error();
    const int rc = check_decode(a);
    return rc ? rc : decode_one((hipStream_t)stream, a);
}

extern "C" int nkv_decode_batch(void* stream, const nkv_decode_args* a, int n) {
    clear_error();
    NKV_REQUIRE(n >= 0 && (n == 0 || a), NKV_ERR_INVALID, "null args");
    bool one = true;
    for (int i = 0; i < n; ++i) {
        const int rc = check_decode(a + i);
        if (rc) return rc;
        const nkv_codec &c = a[i].codec, &f = a[0].codec;
        NKV_REQUIRE(a[i].HD == a[0].HD && c.r == f.r && c.group == f.group &&
                        c.scale_dtype == f.scale_dtype && c.w_dec == f.w_dec && c.mean == f.mean,
                    NKV_ERR_INVALID,
                    "the decodes of one batch must share HD, r, group, scale dtype, w_dec and mean");
        for (int b = 0; b < a[i].B && a[i].rows > 0; ++b)
            one = one && dec_aligned(dec_problem(a + i, b), c.w_dec);
    }
    hipStream_t s = (hipStream_t)stream;
    if (!one) {
        for (int i = 0; i < n; ++i) {
            const int rc = decode_one(s, a + i);
            if (rc) return rc;
        }
        return NKV_OK;
    }
    DecProb p[DEC_MAXB];
    int np = 0;
    for (int i = 0; i < n; ++i) {
        for (int b = 0; b < a[i].B && a[i].rows > 0; ++b) {
            p[np++] = dec_problem(a + i, b);
            if (np == DEC_MAXB) {
                const int rc = launch_decode(s, a, p, np);
                if (rc) return rc;
                np = 0;
            }
        }
    }
    return np ? launch_decode(s, a, p, np) : NKV_OK;
}
