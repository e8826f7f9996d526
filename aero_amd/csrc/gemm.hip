// Quantised GEMM for many tokens on gfx950 (prefill): y[t, r] = sum_c W[r, c] * x[t, c]
// with W in GGML blocks and x, y fp32 — the reference's matmul
// (src/kernels.cpp:520-538) for token counts where re-reading W for every few
// tokens (the GEMV kernels) would dominate. Q8_0 runs gemm_q8_kernel (below);
// the other types gemm_kernel:
//
// A workgroup (4 waves) computes a BM-row x BN-token tile of y. For each
// BK-column chunk of the rows it dequantises its BM rows into LDS as fp32 —
// the reference's dequantised values bit for bit (the arithmetic of
// quant_blocks.hpp) — and stages the BN tokens' x, then each wave runs fp32
// matrix FMAs (v_mfma_f32_16x16x4_f32) over a (BM/2) x (BN/2) sub-tile: exact
// products, fp32 accumulation, so results differ from the reference's serial
// dots only in summation order. The next chunk's weights and x are loaded
// before the current chunk's matrix steps run.
//
// Weight staging: with W 16-byte aligned and rows a multiple of 16 bytes (8
// for IQ4_XS) a thread dequantises one 32-value sub-block per chunk from
// 16-byte loads (2-byte aligned Q6_K blocks are shifted into place
// with byte permutes); otherwise four values at a time from 2- and 4-byte
// loads.
//
// LDS tiles hold element (i, k) of a chunk at i*(BK+4) + (k%4)*(BK/4) + k/4:
// a lane's operands for four consecutive matrix steps (k = 4s + lane/16) are
// one 16-byte read, and the 4-float row pad puts the 16 rows a read touches
// in 16 different bank groups.
//
// HBM bytes per launch: W once per BN-token tile, x once per BM-row tile
// (mostly from L2), y once.
#include "quant_blocks.hpp"

#pragma clang fp contract(off)

namespace aero {

namespace {

struct GemmParams {
    const uint8_t* w;  // n_rows rows of rb bytes
    const float* x;    // n_tok rows of x_stride floats
    float* y;          // n_tok rows of y_stride floats
    int64_t n_rows;
    int n_cols;
    int64_t rb;
    int n_tok;
    int64_t x_stride, y_stride;
};

// ------------------------------------------------- 32-value sub-blocks
// Values c0 .. c0+31 of a row (c0 a multiple of 32), loaded with wide loads
// (load) and dequantised (decode) with the reference's arithmetic.
template <int TYPE> struct Sub32;

// Q4_K (src/kernels.cpp:65-73,337-363): sub-block k = nibble k%2 of qs
// bytes 32(k/2) .. +31; y = (d*sc)*q - (dmin*m).
template <> struct Sub32<AERO_DTYPE_Q4_K> {
    uint4 hd, q[2];
    int k;
    __device__ __forceinline__ void load(const uint8_t* rowp, int c0) {
        const uint8_t* b = rowp + (int64_t)(c0 >> 8) * 144;
        k = (c0 & 255) >> 5;
        hd = ld128(b);
        q[0] = ld128(b + 16 + 32 * (k >> 1));
        q[1] = ld128(b + 32 + 32 * (k >> 1));
    }
    __device__ __forceinline__ void decode(float (&v)[32]) const {
        uint32_t sc, mn;
        kq_scale_min(hd.y, hd.z, hd.w, k, sc, mn);
        const float f = half_bits_to_float(hd.x & 0xFFFFu) * (float)sc;
        const float g = half_bits_to_float(hd.x >> 16) * (float)mn;
        const int sh = (k & 1) ? 4 : 0;
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            const uint32_t w = wd(q, m) >> sh;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[4 * m + e] = f * (float)((w >> (8 * e)) & 15u) - g;
        }
    }
};

// Q5_K (src/kernels.cpp:374-404): Q4_K plus bit k of qh[i] as bit 4.
template <> struct Sub32<AERO_DTYPE_Q5_K> {
    uint4 hd, h[2], q[2];
    int k;
    __device__ __forceinline__ void load(const uint8_t* rowp, int c0) {
        const uint8_t* b = rowp + (int64_t)(c0 >> 8) * 176;
        k = (c0 & 255) >> 5;
        hd = ld128(b);
        h[0] = ld128(b + 16);
        h[1] = ld128(b + 32);
        q[0] = ld128(b + 48 + 32 * (k >> 1));
        q[1] = ld128(b + 64 + 32 * (k >> 1));
    }
    __device__ __forceinline__ void decode(float (&v)[32]) const {
        uint32_t sc, mn;
        kq_scale_min(hd.y, hd.z, hd.w, k, sc, mn);
        const float f = half_bits_to_float(hd.x & 0xFFFFu) * (float)sc;
        const float g = half_bits_to_float(hd.x >> 16) * (float)mn;
        const int sh = (k & 1) ? 4 : 0;
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            const uint32_t w = wd(q, m) >> sh, hb = wd(h, m) >> k;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                v[4 * m + e] =
                    f * (float)(((w >> (8 * e)) & 15u) | (((hb >> (8 * e)) & 1u) << 4)) - g;
        }
    }
};

// Q6_K (src/kernels.cpp:427-458): quarter kq of half h: nibble kq/2 of
// ql[64h + 32(kq%2) + i], bits 2kq of qh[32h + i]; scale sc[8h + 2kq + i/16];
// y = (d*sc)*(q-32). ql and qh from the 48 aligned bytes around each.
template <> struct Sub32<AERO_DTYPE_Q6_K> {
    uint4 l3[3], h3[3];
    uint32_t ph, sc, d;
    int kq;
    __device__ __forceinline__ void load(const uint8_t* rowp, int c0) {
        const uint32_t ob = (uint32_t)(c0 >> 8) * 210u;
        const int h = (c0 >> 7) & 1;
        kq = (c0 >> 5) & 3;
        ph = ob & 15u;
        const uint8_t* b = rowp + (ob - ph);
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            l3[i] = ld128(b + 64 * h + 32 * (kq & 1) + 16 * i);
            h3[i] = ld128(b + 128 + 32 * h + 16 * i);
        }
        sc = ld_u16(rowp + ob + 192 + 8 * h + 2 * kq);
        d = ld_u16(rowp + ob + 208);
    }
    __device__ __forceinline__ void decode(float (&v)[32]) const {
        uint32_t wl[8], wh[8];
        shifted_words<8, 3>(l3, ph, wl);
        shifted_words<8, 3>(h3, ph, wh);
        const float df = half_bits_to_float(d);
        const float f0 = df * (float)(int8_t)(sc & 0xFFu);
        const float f1 = df * (float)(int8_t)((sc >> 8) & 0xFFu);
        const int sl = kq >= 2 ? 4 : 0, shh = 2 * kq;
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            const uint32_t lb = wl[m] >> sl, hb = wh[m] >> shh;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int q = (int)(((lb >> (8 * e)) & 15u) | (((hb >> (8 * e)) & 3u) << 4));
                v[4 * m + e] = (m < 4 ? f0 : f1) * (float)(q - 32);
            }
        }
    }
};

// IQ4_XS (src/kernels.cpp:405-425): sub-block ib: values 0..15 from the low
// nibbles of qs[16ib ..], 16..31 from the high; y = d*(ls-32)*codebook[q].
template <> struct Sub32<AERO_DTYPE_IQ4_XS> {
    uint2 hd, q[2];
    int ib;
    __device__ __forceinline__ void load(const uint8_t* rowp, int c0) {
        const uint8_t* b = rowp + (int64_t)(c0 >> 8) * 136;
        ib = (c0 & 255) >> 5;
        hd = *reinterpret_cast<const uint2*>(b);
        q[0] = *reinterpret_cast<const uint2*>(b + 8 + 16 * ib);
        q[1] = *reinterpret_cast<const uint2*>(b + 16 + 16 * ib);
    }
    __device__ __forceinline__ void decode(float (&v)[32]) const {
        const float d = half_bits_to_float(hd.x & 0xFFFFu);
        const uint32_t sh = hd.x >> 16;
        const uint32_t ls = ((byte_of(hd.y, ib >> 1) >> (4 * (ib & 1))) & 15u) |
                            (((sh >> (2 * ib)) & 3u) << 4);
        const float dl = d * (float)((int)ls - 32);
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            const uint32_t w = (m & 1) ? q[m >> 1].y : q[m >> 1].x;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[4 * m + e] = dl * iq4_level((w >> (8 * e)) & 15u);
                v[16 + 4 * m + e] = dl * iq4_level((w >> (8 * e + 4)) & 15u);
            }
        }
    }
};

// ------------------------------------------------------ weight staging
// FAST: one 32-value sub-block per unit from wide loads (W 16-byte aligned,
// rows a multiple of 16 bytes, 8 for IQ4_XS). Otherwise 16 values per unit,
// four at a time with load_raw / decode.
template <int TYPE, bool FAST, int BM, int BK> struct StageW;

template <int TYPE, int BM, int BK>
struct StageW<TYPE, true, BM, BK> {
    static constexpr int GR = BK / 32;       // sub-blocks per row chunk
    static constexpr int U = BM * GR / 256;  // units per thread
    static_assert(U >= 1 && BM * GR % 256 == 0, "tile");
    Sub32<TYPE> s[U];
    const uint8_t* rowp[U];
    int grp;
    __device__ __forceinline__ void init(const GemmParams& p, int64_t r0, int tid) {
        grp = tid % GR;
#pragma unroll
        for (int u = 0; u < U; ++u)
            rowp[u] = p.w + min(r0 + (tid + 256 * u) / GR, p.n_rows - 1) * p.rb;
    }
    __device__ __forceinline__ void load(const GemmParams&, int kc) {
        const int c = kc * BK + 32 * grp;
#pragma unroll
        for (int u = 0; u < U; ++u) s[u].load(rowp[u], c);
    }
    __device__ __forceinline__ void store(float* As, int tid) const {
        constexpr int RowF = BK + 4;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            float v[32];
            s[u].decode(v);
            float* row = As + ((tid + 256 * u) / GR) * RowF + 8 * grp;
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) {
                *reinterpret_cast<float4*>(row + kk * (BK / 4)) =
                    make_float4(v[kk], v[kk + 4], v[kk + 8], v[kk + 12]);
                *reinterpret_cast<float4*>(row + kk * (BK / 4) + 4) =
                    make_float4(v[kk + 16], v[kk + 20], v[kk + 24], v[kk + 28]);
            }
        }
    }
};

template <int TYPE, int BM, int BK>
struct StageW<TYPE, false, BM, BK> {
    static constexpr int GR = BK / 16;  // 16-value groups per row chunk
    static constexpr int U = BM * GR / 256;
    static_assert(U >= 1 && BM * GR % 256 == 0, "tile");
    using Raw = typename QT<TYPE>::Raw;
    Raw raw[U][4];
    const uint8_t* rowp[U];
    int grp, cc;
    __device__ __forceinline__ void init(const GemmParams& p, int64_t r0, int tid) {
        grp = tid % GR;
#pragma unroll
        for (int u = 0; u < U; ++u)
            rowp[u] = p.w + min(r0 + (tid + 256 * u) / GR, p.n_rows - 1) * p.rb;
    }
    __device__ __forceinline__ void load(const GemmParams&, int kc) {
        cc = kc * BK + 16 * grp;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int cq = cc + 4 * q;
#pragma unroll
            for (int u = 0; u < U; ++u)
                load_raw(rowp[u] + (int64_t)(cq / QT<TYPE>::BV) * QT<TYPE>::BB,
                         (cq % QT<TYPE>::BV) / 4, raw[u][q]);
        }
    }
    __device__ __forceinline__ void store(float* As, int tid) const {
        constexpr int RowF = BK + 4;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            float4 w4[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                w4[q] = decode(raw[u][q], ((cc + 4 * q) % QT<TYPE>::BV) / 4);
            }
            float* row = As + ((tid + 256 * u) / GR) * RowF + 4 * grp;
            *reinterpret_cast<float4*>(row + 0 * BK / 4) = make_float4(w4[0].x, w4[1].x, w4[2].x, w4[3].x);
            *reinterpret_cast<float4*>(row + 1 * BK / 4) = make_float4(w4[0].y, w4[1].y, w4[2].y, w4[3].y);
            *reinterpret_cast<float4*>(row + 2 * BK / 4) = make_float4(w4[0].z, w4[1].z, w4[2].z, w4[3].z);
            *reinterpret_cast<float4*>(row + 3 * BK / 4) = make_float4(w4[0].w, w4[1].w, w4[2].w, w4[3].w);
        }
    }
};

// x staging: 16 consecutive floats of a token per unit.
template <int BN, int BK>
struct StageX {
    static constexpr int GR = BK / 16;
    static constexpr int U = BN * GR / 256;
    static_assert(U >= 1 && BN * GR % 256 == 0, "tile");
    float4 v[U][4];
    const float* xrow[U];
    int grp;
    bool valid;
    __device__ __forceinline__ void init(const GemmParams& p, int t0, int tid) {
        grp = tid % GR;
#pragma unroll
        for (int u = 0; u < U; ++u)
            xrow[u] = p.x + (int64_t)min(t0 + (tid + 256 * u) / GR, p.n_tok - 1) * p.x_stride;
    }
    __device__ __forceinline__ void load(const GemmParams& p, int kc) {
        const int c = kc * BK + 16 * grp;
        valid = c < p.n_cols;
        const int cc = min(c, p.n_cols - 16);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                v[u][q] = *reinterpret_cast<const float4*>(xrow[u] + cc + 4 * q);
    }
    __device__ __forceinline__ void store(float* Bs, int tid) const {
        constexpr int RowF = BK + 4;
        const float4 z = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            float4 x4[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) x4[q] = valid ? v[u][q] : z;
            float* row = Bs + ((tid + 256 * u) / GR) * RowF + 4 * grp;
            *reinterpret_cast<float4*>(row + 0 * BK / 4) = make_float4(x4[0].x, x4[1].x, x4[2].x, x4[3].x);
            *reinterpret_cast<float4*>(row + 1 * BK / 4) = make_float4(x4[0].y, x4[1].y, x4[2].y, x4[3].y);
            *reinterpret_cast<float4*>(row + 2 * BK / 4) = make_float4(x4[0].z, x4[1].z, x4[2].z, x4[3].z);
            *reinterpret_cast<float4*>(row + 3 * BK / 4) = make_float4(x4[0].w, x4[1].w, x4[2].w, x4[3].w);
        }
    }
};

// ---------------------------------------------------------------- kernel
// 4 waves in a 2 x 2 grid, each owning (BM/2) x (BN/2) as 16 x 16 tiles.
template <int TYPE, bool FAST, int BM, int BN, int BK>
__global__ __launch_bounds__(256) void gemm_kernel(GemmParams p) {
    constexpr int RowF = BK + 4;               // floats per padded LDS tile row
    constexpr int MI = BM / 32, NI = BN / 32;  // matrix tiles per wave
    __shared__ __align__(16) float As[BM * RowF];
    __shared__ __align__(16) float Bs[BN * RowF];

    const int tid = threadIdx.x;
    const int l = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave & 1, wn = wave >> 1;
    const int64_t r0 = (int64_t)blockIdx.x * BM;
    const int t0 = blockIdx.y * BN;
    const int n_k = (p.n_cols + BK - 1) / BK;

    v4f acc[MI][NI];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

    StageW<TYPE, FAST, BM, BK> sw;
    StageX<BN, BK> sx;
    sw.init(p, r0, tid);
    sx.init(p, t0, tid);

    sx.load(p, 0);
    sw.load(p, 0);
    sw.store(As, tid);
    sx.store(Bs, tid);
    __syncthreads();
    const float* ap = As + ((BM / 2) * wm + (l & 15)) * RowF + (l >> 4) * (BK / 4);
    const float* bp = Bs + ((BN / 2) * wn + (l & 15)) * RowF + (l >> 4) * (BK / 4);
    for (int kc = 0; kc < n_k; ++kc) {
        // the next chunk's loads go out before this chunk's matrix steps
        const int kn = min(kc + 1, n_k - 1);
        sx.load(p, kn);
        sw.load(p, kn);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int sg = 0; sg < BK / 16; ++sg) {
            float4 a[MI], b[NI];
#pragma unroll
            for (int i = 0; i < MI; ++i)
                a[i] = *reinterpret_cast<const float4*>(ap + 16 * i * RowF + 4 * sg);
#pragma unroll
            for (int j = 0; j < NI; ++j)
                b[j] = *reinterpret_cast<const float4*>(bp + 16 * j * RowF + 4 * sg);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < MI; ++i)
#pragma unroll
                    for (int j = 0; j < NI; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][e], b[j][e],
                                                                         acc[i][j], 0, 0, 0);
        }
        if (kc + 1 >= n_k) break;
        __syncthreads();  // every wave is done reading this chunk
        sw.store(As, tid);
        sx.store(Bs, tid);
        __syncthreads();
    }

    // acc[i][j] holds rows 4(l/16)+v, token l%16 of matrix tile (i, j)
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) {
            const int64_t row = r0 + (BM / 2) * wm + 16 * i + 4 * (l >> 4);
            const int tok = t0 + (BN / 2) * wn + 16 * j + (l & 15);
            if (tok < p.n_tok) {
                float* yp = p.y + (int64_t)tok * p.y_stride;
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    if (row + v < p.n_rows) yp[row + v] = acc[i][j][v];
            }
        }
}

// ------------------------------------------------------- Q8_0, bf16 parts
// y[t, r] = sum_b d_b sum_c q_c x_c over Q8_0 blocks b of 32: a matrix step of
// v_mfma_f32_16x16x32_bf16 covers one block of 16 rows and 16 tokens. int8
// codes are exact in bf16, and x is the exact sum of three bf16 parts (its 24
// bits cut after 8 and 16), so every product is exact; a block's three steps,
// the smallest part first, are summed in fp32 from zero and added to the
// row's sum times d, one rounding a block. (D holds tokens 4(l/16) + v of row
// l%16: d is lane-local. Lane l supplies columns 8(l/16) .. +7 of token l%16
// and of row l%16, loaded as they lie.)
//
// d comes after the sum over the block, and the smallest part of an x below
// 2^-110 is below bf16's last bit: a step whose x lies outside 2^-100 .. 2^100
// is computed on x times a power of two a token.
//
// The eight waves of a workgroup own the same NT x 16 rows and MT x 16 tokens
// and take every eighth block; their sums meet in LDS once at the end, so
// the loop has no barrier and no LDS traffic, and short rows (896 columns: 28
// blocks) still keep eight waves busy. A part of x costs vector instructions
// per row tile instead (about as long as the matrix steps at NT = 2).
// Measured on MI355X against the fp32 matrix steps of gemm_kernel (2.7 times
// the matrix time, 128-column chunks between barriers): see launch_q8.
constexpr uint32_t kQ8Large = 227u << 23, kQ8Small = 27u << 23;   // 2^100, 2^-100
typedef __bf16 bf8v __attribute__((ext_vector_type(8)));

// 8 int8 codes (two dwords) as bf16: each byte offset by 128, converted and
// shifted back (exact), the upper halves of the floats packed
__device__ __forceinline__ bf8v q8_bf16(uint32_t w0, uint32_t w1) {
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const uint32_t u = (i ? w1 : w0) ^ 0x80808080u;
        const float f0 = (float)(u & 255u) - 128.0f, f1 = (float)((u >> 8) & 255u) - 128.0f;
        const float f2 = (float)((u >> 16) & 255u) - 128.0f, f3 = (float)(u >> 24) - 128.0f;
        o[2 * i] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, f1),
                                         __builtin_bit_cast(uint32_t, f0), 0x07060302u);
        o[2 * i + 1] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, f3),
                                             __builtin_bit_cast(uint32_t, f2), 0x07060302u);
    }
    return __builtin_bit_cast(bf8v, make_uint4(o[0], o[1], o[2], o[3]));
}

// 8 floats as three bf16 parts (part 0 the largest); with INF an infinity
// keeps part 0 alone
template <bool INF>
__device__ __forceinline__ void bf16_parts(const float (&x)[8], bf8v (&p)[3]) {
    float r[3][8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float h = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, x[i]) & 0xFFFF0000u);
        r[0][i] = h;
        r[1][i] = x[i] - h;
        const float m =
            __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, r[1][i]) & 0xFFFF0000u);
        r[2][i] = r[1][i] - m;
        if (INF && fabsf(x[i]) > 3.4028235e38f) r[1][i] = r[2][i] = 0.0f;
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        uint32_t o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            o[i] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, r[k][2 * i + 1]),
                                         __builtin_bit_cast(uint32_t, r[k][2 * i]), 0x07060302u);
        p[k] = __builtin_bit_cast(bf8v, make_uint4(o[0], o[1], o[2], o[3]));
    }
}

// the largest magnitude of 8 floats (a NaN is ignored: it shows in the sums)
__device__ __forceinline__ float largest(const float (&x)[8]) {
    float big = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; i += 2)
        asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(big) : "v"(x[i]), "v"(x[i + 1]));
    return big;
}

constexpr int kQ8Waves = 8;

template <int MT, int NT>
__global__ __launch_bounds__(64 * kQ8Waves) void gemm_q8_kernel(GemmParams p) {
    __shared__ v4f sums[kQ8Waves][MT * NT][64];
    const int l = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c = l & 15, g = l >> 4;
    const int64_t r0 = (int64_t)blockIdx.x * (16 * NT);
    const int t0 = blockIdx.y * (16 * MT);
    const int nb = p.n_cols / 32;

    // lane's rows and tokens (clamped: the copies are not stored)
    const uint8_t* wp[NT];
    const float* xp[MT];
#pragma unroll
    for (int j = 0; j < NT; ++j)
        wp[j] = p.w + min(r0 + 16 * j + c, p.n_rows - 1) * p.rb;
#pragma unroll
    for (int m = 0; m < MT; ++m)
        xp[m] = p.x + (int64_t)min(t0 + 16 * m + c, p.n_tok - 1) * p.x_stride + 8 * g;

    v4f xa[MT][2];
    uint32_t wq[NT][3];
    uint32_t wd[NT];
    // the codes lie 2 bytes off a dword in every other block (and row, where
    // their number is odd): two dwords from the one that holds the first code,
    // and the last two codes, which lie in neither there; shifted into place
    auto load = [&](int b) __attribute__((always_inline)) {
        b = min(b, nb - 1);
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            xa[m][0] = *reinterpret_cast<const v4f*>(xp[m] + 32 * b);
            xa[m][1] = *reinterpret_cast<const v4f*>(xp[m] + 32 * b + 4);
        }
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const uint8_t* e = wp[j] + (int64_t)34 * b;
            const uintptr_t a = reinterpret_cast<uintptr_t>(e + 2 + 8 * g);
            const uint32_t* d = reinterpret_cast<const uint32_t*>(a & ~uintptr_t(3));
            wq[j][0] = d[0];
            wq[j][1] = d[1];
            wq[j][2] = *reinterpret_cast<const uint16_t*>(e + 8 + 8 * g);
            wd[j] = *reinterpret_cast<const uint16_t*>(e);
        }
    };

    v4f acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[m][j] = v4f{0.f, 0.f, 0.f, 0.f};

    load(wave);
    for (int b = wave; b < nb; b += kQ8Waves) {
        bf8v wb[NT];
        float d[NT];
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const uint32_t sh = (uint32_t)(reinterpret_cast<uintptr_t>(wp[j] + (int64_t)34 * b + 2) & 2);
            wb[j] = q8_bf16(__builtin_amdgcn_alignbyte(wq[j][1], wq[j][0], sh),
                            __builtin_amdgcn_alignbyte(wq[j][2], wq[j][1], sh));
            d[j] = half_bits_to_float(wd[j]);
        }
        float x[MT][8];
        uint32_t hi = 0, lo = ~0u;    // bits of the largest values; zeros pass
#pragma unroll
        for (int m = 0; m < MT; ++m) {
#pragma unroll
            for (int i = 0; i < 8; ++i) x[m][i] = xa[m][i >> 2][i & 3];
            const uint32_t u = __builtin_bit_cast(uint32_t, largest(x[m]));
            hi = max(hi, u);
            lo = min(lo, u - 1);
        }
        bf8v xb[MT][3];
        auto product = [&](int m, int j) __attribute__((always_inline)) {
            v4f part = {0.f, 0.f, 0.f, 0.f};
            part = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xb[m][2], wb[j], part, 0, 0, 0);
            part = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xb[m][1], wb[j], part, 0, 0, 0);
            return __builtin_amdgcn_mfma_f32_16x16x32_bf16(xb[m][0], wb[j], part, 0, 0, 0);
        };
        if (!__any(hi > kQ8Large || lo < kQ8Small)) {
#pragma unroll
            for (int m = 0; m < MT; ++m) bf16_parts<false>(x[m], xb[m]);
            load(b + kQ8Waves);
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    const v4f part = product(m, j);
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        acc[m][j][v] = __builtin_fmaf(part[v], d[j], acc[m][j][v]);
                }
        } else {
            // a token's 32 values times the power of two 2^-e that brings
            // the largest near 1; half of 2^e goes to the sum, half to d
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                uint32_t t = __builtin_bit_cast(uint32_t, largest(x[m]));
                t = max(t, (uint32_t)__shfl_xor((int)t, 16));
                t = max(t, (uint32_t)__shfl_xor((int)t, 32));
                const int e = (int)(t >> 23) - 126;
#pragma unroll
                for (int i = 0; i < 8; ++i) x[m][i] = ldexpf(x[m][i], -e);
                bf16_parts<true>(x[m], xb[m]);
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    const v4f part = product(m, j);
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const int ev = __shfl(e, 4 * g + v);
                        acc[m][j][v] = __builtin_fmaf(ldexpf(part[v], ev / 2),
                                                      ldexpf(d[j], ev - ev / 2), acc[m][j][v]);
                    }
                }
            }
            load(b + kQ8Waves);
        }
    }

#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int j = 0; j < NT; ++j) sums[wave][m * NT + j][l] = acc[m][j];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MT * NT; i += kQ8Waves) {
        if (i + wave >= MT * NT) break;
        const int m = (i + wave) / NT, j = (i + wave) % NT;
        v4f y = sums[0][i + wave][l];
#pragma unroll
        for (int k = 1; k < kQ8Waves; ++k) y += sums[k][i + wave][l];
        const int64_t row = r0 + 16 * j + c;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int tok = t0 + 16 * m + 4 * g + v;
            if (row < p.n_rows && tok < p.n_tok) p.y[(int64_t)tok * p.y_stride + row] = y[v];
        }
    }
}

using GemmKernel = void (*)(GemmParams);

template <bool FAST>
GemmKernel pick_gemm(int dtype) {
    constexpr int BM = 64, BN = 64, BK = 128;
    switch (dtype) {
    case AERO_DTYPE_Q4_K: return gemm_kernel<AERO_DTYPE_Q4_K, FAST, BM, BN, BK>;
    case AERO_DTYPE_Q5_K: return gemm_kernel<AERO_DTYPE_Q5_K, FAST, BM, BN, BK>;
    case AERO_DTYPE_Q6_K: return gemm_kernel<AERO_DTYPE_Q6_K, FAST, BM, BN, BK>;
    case AERO_DTYPE_IQ4_XS: return gemm_kernel<AERO_DTYPE_IQ4_XS, FAST, BM, BN, BK>;
    default: return nullptr;
    }
}

}  // namespace

namespace {

// A workgroup tile of gemm_q8_kernel and its cost a block step with one
// workgroup a CU (measured on MI355X, us for eight waves taking a block each,
// 896 x 4864; there is no term for memory or for small tiles that share a CU.
// Over rows of 2816 to 7424 columns and 4 to 1300 tokens calls took 1.0 to 1.4
// times their tile's cost, the more the smaller, plus 1 to 3 us.)
struct Q8Tile {
    int mt, nt;
    double cost;
    void (*k)(GemmParams);
};
const Q8Tile kQ8Tiles[] = {
    {1, 1, 0.65, gemm_q8_kernel<1, 1>}, {2, 1, 1.05, gemm_q8_kernel<2, 1>},
    {1, 2, 1.15, gemm_q8_kernel<1, 2>}, {2, 2, 1.50, gemm_q8_kernel<2, 2>},
    {4, 2, 2.35, gemm_q8_kernel<4, 2>}, {2, 4, 2.50, gemm_q8_kernel<2, 4>},
    {4, 4, 3.30, gemm_q8_kernel<4, 4>},
};

// The tile whose rounds of one workgroup a CU cost least (the waves' longest
// share of a row's blocks apart). Measured on MI355X, fp32-step GEMM (GEMV
// below 32 tokens) / this in us: 4864 x 896 at 8 tokens 13.8 / 6.4, 32 30.6 /
// 8.2, 77 31.8 / 12.5, 512 75.8 / 44.5; 896 x 4864 at 77 116 / 25.1; 4096 x
// 4096 at 512 171 / 152; 14336 x 4096 at 64 100.5 / 77.7, 512 577 / 522. Error
// against float64 at 896 columns 5.3e-7 -> 7.6e-8.
const Q8Tile& q8_tile(int64_t n_rows, int64_t n_tok, double* cost = nullptr) {
    const int64_t cus = cu_count();
    const Q8Tile* best = nullptr;
    double least = 0.0;
    for (const Q8Tile& t : kQ8Tiles) {
        const int64_t tt = (n_tok + 16 * t.mt - 1) / (16 * t.mt);
        const int64_t wgs = (n_rows + 16 * t.nt - 1) / (16 * t.nt) * tt;
        // (the last tile takes any call that gemm_dev admits)
        if (tt > 65535 && &t != std::end(kQ8Tiles) - 1) continue;
        const double c = (double)((wgs + cus - 1) / cus) * t.cost;
        if (best == nullptr || c < least) {
            best = &t;
            least = c;
        }
    }
    if (cost != nullptr) *cost = least;
    return *best;
}

// (AERO_HIP_TUNE gemm_q8_tile=N takes entry N - 1 instead.)
bool launch_q8(const GemmParams& p, hipStream_t s) {
    const Q8Tile* best = &q8_tile(p.n_rows, p.n_tok);
    const int fixed = tune("gemm_q8_tile", 0);
    if (fixed >= 1 && fixed <= (int)(sizeof(kQ8Tiles) / sizeof(kQ8Tiles[0])))
        best = &kQ8Tiles[fixed - 1];
    const int64_t rt = (p.n_rows + 16 * best->nt - 1) / (16 * best->nt);
    const int64_t tt = ((int64_t)p.n_tok + 16 * best->mt - 1) / (16 * best->mt);
    return launch("gemm_q8_kernel", best->k, dim3((unsigned)rt, (unsigned)tt),
                  dim3(64 * kQ8Waves), 0, s, p);
}

}  // namespace

double q8_gemm_cost(int64_t n_rows, int64_t n_tok) {
    double c = 0.0;
    q8_tile(n_rows, n_tok, &c);
    return c;
}

// Called by gemv_dev after its argument checks (W's size and 4-byte
// alignment, x 16-byte aligned, n_cols a multiple of the block), for
// launches of many tokens.
bool gemm_dev(int dtype, const uint8_t* w, const float* x, float* y, int64_t n_rows,
              int64_t n_cols, int64_t rb, int64_t n_tok, hipStream_t s) {
    const int64_t row_tiles = (n_rows + 63) / 64, tok_tiles = (n_tok + 63) / 64;
    const bool fast = dtype == AERO_DTYPE_IQ4_XS
                          ? (reinterpret_cast<uintptr_t>(w) & 7u) == 0 && rb % 8 == 0
                          : aligned16(w) && rb % 16 == 0;
    const GemmParams p{w, x, y, n_rows, (int)n_cols, rb, (int)n_tok, n_cols, n_rows};
    if (dtype == AERO_DTYPE_Q8_0 && row_tiles <= 0x1fffffff && tok_tiles <= 65535)
        return launch_q8(p, s);
    GemmKernel k = (fast && tune("gemm_fast", 1)) ? pick_gemm<true>(dtype) : pick_gemm<false>(dtype);
    if (k == nullptr || row_tiles > 0x7fffffff || tok_tiles > 65535 || n_cols % 32 != 0) {
        set_error("matmul: no GEMM for dtype %d at %lld x %lld, %lld tokens", dtype,
                  (long long)n_rows, (long long)n_cols, (long long)n_tok);
        return false;
    }
    return launch("gemm_kernel", k, dim3((unsigned)row_tiles, (unsigned)tok_tiles), dim3(256), 0,
                  s, p);
}

}  // namespace aero
