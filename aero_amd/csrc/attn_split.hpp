// Prefill attention over an fp32 KV cache on the fp16 matrix cores (included
// by attention.hip after its fp16 helpers).
//
// v_mfma_f32_32x32x16_f16: lane l (n = l % 32, h = l / 32) supplies
// A[n][8h..8h+7] and B[8h..8h+7][n] and receives D[8j + 4h + r][n], j, r =
// 0..3, in element 4j + r. Everything is computed transposed, so a lane's
// column is one query throughout and the softmax state, its rescaling and the
// output rows are lane-local:
//  * S^T = K Q^T: A = 32 keys x 16 dimensions, B = the wave's 32 queries;
//  * O^T += V^T P^T: A = 32 value dimensions x 16 keys, B = the
//    probabilities as the scores' accumulator holds them (k-slots 8h + 4b + r
//    of step s are key 16s + 8b + 4h + r, and V^T is stored in that order).
// The waves share the keys of a tile; a group of queries is 32 vectors.
//
// Arithmetic: q (a power of two per query), K and V (a power of two per
// wave's share of a tile, KW keys) are scaled to below 2^14 and split into
// two fp16 parts, hi = fp16(v), lo = fp16(v - hi): 22 bits, and 2^-39 of the
// block's largest below that. Products are hi hi + hi lo + lo hi, exact,
// added in fp32 by the matrix cores. The probabilities (<= 1, against a
// reference max m that is a whole number of log2 units) are split the same
// way, in units of 2^(ev - E + 14), ev the exponent of the key's V block and E
// that of the sums; the sums take each step's product with one fma, which
// carries the change of m and E. Keys that no query of the workgroup
// keeps become zeros, so what lies in them does not touch the scales.
// What the split cannot carry ends the walk, and the workgroup does its 128
// rows again on fp32 matrix steps (attn_tile_fp32, the sums of
// attn_mfma_kernel): an infinity (a split makes a NaN of it), sums that are
// not finite (a NaN among the values reaches queries that do not keep its
// key), rows of V whose exponents differ by more than kSpread, in a block or
// between blocks (a query may keep the small ones alone), dimensions of V that
// do by more than kSpreadCh (known at the end of the walk), or keys and queries
// whose products pass 2^kScoreExp. Time of calls whose every workgroup does
// so, fp32-step kernel / this one (where the end of the walk shows it), 2048
// causal tokens: 32 / 8 heads of dim 128 470 / 511 us (670), of dim 64 274 / 341 us
// (419), 8 / 4 heads of dim 256 in a window of 1024, whose 128 workgroups leave
// half of the CUs idle, 240 / 647 us (780).
//
// Precision. An operand keeps 22 to 23 bits and the lo lo products are
// dropped, where the fp32 steps keep 24; the sums are shorter and exact in the
// rescaling. 2-norm error against float64, normal q, K and V, is below the
// fp32 steps' at every size measured (below; 33 queries of dim 128 1.8e-7 ->
// 1.6e-7, 1641 of dim 256 5.4e-7 -> 3.8e-7); where all probabilities are
// nearly the same, which rounds least in fp32, above (0.8e-7 -> 1.1e-7). It is
// an error relative to the query's largest values of V: an element far below
// the others of its query has fewer bits.
//
// Shape. A workgroup owns 128 query vectors of one kv head (32 a wave). At
// head dims 64 and 128 eight waves walk 128 / 64 keys a step, two waves a
// query group, each on half of the sub-tiles (their sums meet in LDS at the
// end): a workgroup's walk, which bounds the call where the causal triangle
// leaves some twice the mean, is half as long as with four. At 256 the
// query's parts and the sums take 256 registers, so four waves with the
// register file to themselves walk 32 keys. K and V are split once a
// workgroup into LDS (double-buffered; the split runs between the scores'
// matrix steps, the next loads between the value sum's).
// What bounds it: per 64 keys and CU at head dim 128 3072 cycles of matrix
// steps a SIMD, about 2600 of LDS, about 2400 of vector instructions a SIMD
// and a step takes about 7500: two waves a SIMD (all 256 registers each) do
// not overlap them fully (92 bytes a lane do not fit at head dim 128, 104 with
// key positions: four vectors of q's parts come from scratch each step, between
// the scores' matrix steps). Against attn_mfma_kernel, whose fp32 steps run at a
// sixteenth of the fp16 rate, on MI355X, 2048 causal tokens: 32 / 8 heads of
// dim 128 455 -> 150 us (229 TFLOP/s by the useful products), of dim 64
// 247 -> 95 us, 8 / 4 heads of dim 256 in a window of 1024 207 -> 148 us.
// Error against float64 (2-norm) at those sizes: 4.0e-7 -> 2.9e-7, 3.3e-7 ->
// 2.5e-7, 5.0e-7 -> 3.5e-7.

typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v2f __attribute__((ext_vector_type(2)));

template <int D>
struct SplitCfg {
    static constexpr int NW = D == 256 ? 4 : 8;       // waves
    static constexpr int GK = NW / 4;                 // waves on the same queries
    static constexpr int KT = D == 64 ? 128 : (D == 128 ? 64 : 32);   // keys a tile
    static constexpr int SUBS = KT / 32;
    static constexpr int KW = KT / NW;                // keys a wave converts
    static constexpr int LK = D / 8;                  // K: lanes a key (8 dimensions each)
    static constexpr int PK = 64 / LK, NK = KW / PK;  // keys a pass, passes
    static constexpr int CV = D == 256 ? 2 : 1;       // V: column passes (2 dimensions a lane)
    static constexpr int NP = NK + 2 * CV;            // pieces of 8 elements a lane converts
    static constexpr int OW = KW / 8;                 // key octets a wave converts
    static constexpr int KP = D + 8;                  // K row pitch, halves
    static constexpr int VP = 40;                     // V^T row pitch, halves (32 keys + 16 B)
    static constexpr int KPART = KT * KP, VPART = SUBS * D * VP;
    static constexpr int BUF = 2 * (KPART + VPART);   // halves
};

// two fp32 values (already scaled) as fp16 hi and lo pairs: lo from one
// mixed-precision fma an element (v_fma_mix_f32 issues in half the time of
// v_fma_mixlo_f16, which the compiler prefers) and a packed conversion
__device__ __forceinline__ void split_pair(float a, float b, h2& hi, h2& lo) {
    hi = __builtin_convertvector((v2f){a, b}, h2);
    float x, y;
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(x) : "v"(hi), "v"(a));
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]"
        : "=v"(y) : "v"(hi), "v"(b));
    lo = __builtin_convertvector((v2f){x, y}, h2);
}

// max of three (magnitudes): v_max3_f32 directly, without the compiler's
// quieting of each operand (a NaN is ignored; it shows in the results)
__device__ __forceinline__ float max3(float a, float b, float c) {
    asm("v_max3_f32 %0, %0, %1, %2" : "+v"(a) : "v"(b), "v"(c));
    return a;
}
__device__ __forceinline__ float max3_abs(float a, float b, float c) {
    asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(a) : "v"(b), "v"(c));
    return a;
}
__device__ __forceinline__ float min3_abs(float a, float b, float c) {
    asm("v_min3_f32 %0, |%0|, |%1|, |%2|" : "+v"(a) : "v"(b), "v"(c));
    return a;
}

// the largest a and b over each 16-lane row, in every lane of it (a DPP
// operand may be read two instructions after it is written)
__device__ __forceinline__ void row_max2(float& a, float& b) {
    asm("s_nop 1\n"
        "v_max_f32_dpp %0, %0, %0 row_ror:8 row_mask:0xf bank_mask:0xf\n"
        "v_max_f32_dpp %1, %1, %1 row_ror:8 row_mask:0xf bank_mask:0xf\n"
        "s_nop 0\n"
        "v_max_f32_dpp %0, %0, %0 row_ror:4 row_mask:0xf bank_mask:0xf\n"
        "v_max_f32_dpp %1, %1, %1 row_ror:4 row_mask:0xf bank_mask:0xf\n"
        "s_nop 0\n"
        "v_max_f32_dpp %0, %0, %0 row_ror:2 row_mask:0xf bank_mask:0xf\n"
        "v_max_f32_dpp %1, %1, %1 row_ror:2 row_mask:0xf bank_mask:0xf\n"
        "s_nop 0\n"
        "v_max_f32_dpp %0, %0, %0 row_ror:1 row_mask:0xf bank_mask:0xf\n"
        "v_max_f32_dpp %1, %1, %1 row_ror:1 row_mask:0xf bank_mask:0xf\n"
        "s_nop 1"
        : "+v"(a), "+v"(b));
}
__device__ __forceinline__ float lane_value(float x, int lane) {
    return __builtin_bit_cast(float,
                              __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), lane));
}
// the same for each half of the wave, in its lane 31 (row 1 has met row 0)
__device__ __forceinline__ void half_max2(float& a, float& b) {
    row_max2(a, b);
    asm("v_max_f32_dpp %0, %0, %0 row_bcast:15 row_mask:0xa bank_mask:0xf\n"
        "v_max_f32_dpp %1, %1, %1 row_bcast:15 row_mask:0xa bank_mask:0xf\n"
        "s_nop 1"
        : "+v"(a), "+v"(b));
}
// the largest a and b over the wave, wave-uniform
__device__ __forceinline__ void wave_max2(float& a, float& b) {
    row_max2(a, b);
    asm("v_max_f32_dpp %0, %0, %0 row_bcast:15 row_mask:0xa bank_mask:0xf\n"
        "v_max_f32_dpp %1, %1, %1 row_bcast:15 row_mask:0xa bank_mask:0xf\n"
        "s_nop 0\n"
        "v_max_f32_dpp %0, %0, %0 row_bcast:31 row_mask:0xc bank_mask:0xf\n"
        "v_max_f32_dpp %1, %1, %1 row_bcast:31 row_mask:0xc bank_mask:0xf\n"
        "s_nop 1"
        : "+v"(a), "+v"(b));
    a = lane_value(a, 63);
    b = lane_value(b, 63);
}

// e with |x| < 2^e for a block's largest |x|, clamped so that 2^(14 - e) and
// 2^(e - 14) are normal (129 for an infinity)
__device__ __forceinline__ int block_exp(float amax) {
    return max((int)(__builtin_bit_cast(uint32_t, amax) >> 23) - 126, -112);
}

// One wave's n query vectors u0.. of kv head kh over keys [j0, j1), one after
// the other in plain fp32, so that a value that is not finite reaches only the
// queries that keep its key. 64 keys a step, a lane a key for the scores, a
// lane D / 64 dimensions for the value sum.
template <int D>
__device__ __forceinline__ void attn_rows_plain(const AttnParams& p, int64_t u0, int n, int kh,
                                                int j0, int j1) {
    constexpr int E = D / 64;
    const int lane = threadIdx.x & 63;
    const float* kg = static_cast<const float*>(p.k);
    const float* vg = static_cast<const float*>(p.v);
    for (int i = 0; i < n; ++i) {
        const int64_t u = u0 + i, t = u / p.rep;
        const int64_t row = t * p.n_head + (int64_t)kh * p.rep + u % p.rep;
        const int64_t qp = p.qpos ? (int64_t)p.qpos[t] : t;
        const float* q = p.q + row * D;
        float m = -INFINITY, l = 0.0f, acc[E];
        for (int e = 0; e < E; ++e) acc[e] = 0.0f;
        for (int jb = j0; jb < j1; jb += 64) {
            const int j = min(jb + lane, j1 - 1);
            const float* kv = kg + ((int64_t)j * p.n_head_kv + kh) * D;
            float s = 0.0f;
#pragma unroll 4
            for (int d = 0; d < D; ++d) s = __builtin_fmaf(q[d], kv[d], s);
            const int64_t kp = p.kpos ? (int64_t)p.kpos[j] : j;
            const bool keep = jb + lane < j1 && key_kept(kp, qp, p.window);
            s = keep ? s * p.scale : -INFINITY;
            float mn = fmaxf(m, s);
            for (int off = 32; off >= 1; off >>= 1) mn = fmaxf(mn, __shfl_xor(mn, off));
            const float alpha = (m == -INFINITY) ? 0.0f : expf(m - mn);
            const float pr = (s == -INFINITY) ? 0.0f : expf(s - mn);
            l = l * alpha + group_sum<64>(pr);
            for (int e = 0; e < E; ++e) acc[e] *= alpha;
            for (uint64_t left = __ballot(keep); left != 0; left &= left - 1) {
                const int x = __ffsll((unsigned long long)left) - 1;
                const float w = __shfl(pr, x);
                const float* vv = vg + ((int64_t)(jb + x) * p.n_head_kv + kh) * D;
                for (int e = 0; e < E; ++e)
                    acc[e] = __builtin_fmaf(w, vv[64 * e + lane], acc[e]);
            }
            m = mn;
        }
        for (int e = 0; e < E; ++e) p.out[row * D + 64 * e + lane] = acc[e] / fmaxf(l, 1e-30f);
    }
}

// Four waves' 16-query tile (query vectors 16 tile .. of kv head kh) over all
// its keys on the fp32 matrix cores, as attn_mfma_kernel computes it: wave w
// takes every fourth 16-key tile, the sums meet in LDS (sums; calls are
// bracketed by barriers, so every wave of the workgroup makes as many). Where
// a key tile holds keys that some of the queries do not keep, a value that is
// not finite would reach those too (0 times it): such a query tile is done in
// plain fp32.
template <int D>
struct TileSums {
    float m[4][16], l[4][16];
    int leak[4];
    float acc[4][16][D + 4];
};

template <int D>
__device__ __forceinline__ void attn_tile_fp32(const AttnParams& p, int64_t tile, int kh,
                                               TileSums<D>& sums) {
    using Tile = KvTile<0, D, D>;
    constexpr int KS = Tile::KS, VS = Tile::VS;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));   // (apart from the walk's lane: no register held for it)
    tid &= 255;
    const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, c = lane & 15;
    const int64_t n_vec = p.n_q * p.rep, u0 = tile * 16;
    const int64_t u = u0 + c;
    const bool qok = u < n_vec;
    const int64_t uc = qok ? u : n_vec - 1;
    const int64_t tq = uc / p.rep;
    const int64_t qrow = tq * p.n_head + (int64_t)kh * p.rep + uc % p.rep;
    const int64_t qp = p.qpos ? (int64_t)p.qpos[tq] : tq;
    float qs[KS];
#pragma unroll
    for (int e = 0; e < KS; e += 4) {
        const v4f f = *reinterpret_cast<const v4f*>(p.q + qrow * D + Tile::kdim(g, e));
#pragma unroll
        for (int x = 0; x < 4; ++x) qs[e + x] = qok ? f[x] : 0.0f;
    }
    int64_t i_lo = 0, i_hi = u0 < n_vec ? (p.n_kv + 15) / 16 : 0;
    if (p.kpos == nullptr) {
        int64_t qmin = qp, qmax = qp;
#pragma unroll
        for (int off = 8; off >= 1; off >>= 1) {
            qmin = min(qmin, (int64_t)__shfl_xor(qmin, off, 16));
            qmax = max(qmax, (int64_t)__shfl_xor(qmax, off, 16));
        }
        i_hi = min(i_hi, max<int64_t>(0, (qmax + 16) / 16));
        if (p.window > 0) i_lo = max<int64_t>(0, (qmin - p.window + 1) / 16);
    }
    float m = -INFINITY, ls = 0.0f;
    v4f acc[VS];
#pragma unroll
    for (int t = 0; t < VS; ++t) acc[t] = v4f{0.f, 0.f, 0.f, 0.f};
    bool leak = false;
    for (int64_t i = i_lo + w; i < i_hi; i += 4) {
        Tile tl;
        tl.load(p, 16 * i, p.n_kv, g, c, kh);
        bool part = false;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int64_t kj = 16 * i + 4 * g + r;
            const int64_t kp = p.kpos ? (int64_t)__shfl(tl.kp, 4 * g + r) : kj;
            part = part || (qok && !(kj < p.n_kv && key_kept(kp, qp, p.window)));
        }
        if (__any(part)) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int t = 0; t < VS; ++t)
                    leak = leak || !(fabsf(slice_elem<0>(tl.v[r], t)) <= 3.4028235e38f);
        }
        mfma_step<0, D, D>(p, tl, qs, 16 * i, p.n_kv, qp, qok, g, m, ls, acc);
    }
    ls += __shfl_xor(ls, 16);
    ls += __shfl_xor(ls, 32);
    if (g == 0) {
        sums.m[w][c] = m;
        sums.l[w][c] = ls;
    }
    leak = __any(leak);
    if (lane == 0) sums.leak[w] = leak;
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int t = 0; t < VS; t += 4)
            *reinterpret_cast<v4f*>(&sums.acc[w][4 * g + r][Tile::vdim(c, t)]) =
                v4f{acc[t][r], acc[t + 1][r], acc[t + 2][r], acc[t + 3][r]};
    __syncthreads();
    if (sums.leak[0] | sums.leak[1] | sums.leak[2] | sums.leak[3]) {
        attn_rows_plain<D>(p, u0 + 4 * w, (int)max<int64_t>(0, min<int64_t>(4, n_vec - u0 - 4 * w)),
                           kh, (int)(16 * i_lo), (int)min<int64_t>(16 * i_hi, p.n_kv));
        return;
    }
    // thread (query tid / 16, 4 value elements at a time)
    const int qi = tid >> 4;
    if (u0 + qi >= n_vec) return;
    const int64_t row = (u0 + qi) / p.rep * p.n_head + (int64_t)kh * p.rep + (u0 + qi) % p.rep;
    float mt = -INFINITY, lt = 0.0f, sc[4];
#pragma unroll
    for (int x = 0; x < 4; ++x) mt = fmaxf(mt, sums.m[x][qi]);
#pragma unroll
    for (int x = 0; x < 4; ++x) {
        sc[x] = sums.m[x][qi] == -INFINITY ? 0.0f : expf(sums.m[x][qi] - mt);
        lt += sums.l[x][qi] * sc[x];
    }
    lt = fmaxf(lt, 1e-30f);
#pragma unroll 1
    for (int d = 4 * (tid & 15); d < D; d += 64) {
        v4f o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            const v4f a = *reinterpret_cast<const v4f*>(&sums.acc[x][qi][d]);
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = __builtin_fmaf(a[e], sc[x], o[e]);
        }
        *reinterpret_cast<v4f*>(p.out + row * D + d) = v4f{o[0] / lt, o[1] / lt, o[2] / lt, o[3] / lt};
    }
}

constexpr float kLog2eLo = 1.92596299e-8f;   // log2(e) - kLog2e
constexpr int kNoMax = -(1 << 28);     // no key kept yet
constexpr int kSplitVecs = 128;   // query vectors a workgroup
// Largest difference of the exponents of two rows of V that a workgroup may
// keep. A query may keep small rows alone, or large ones with probabilities
// that make them as small: what the parts drop, 2^-39 of the largest, is then
// 2^-21 of the query's result, which is what the fp32 steps' sums leave.
constexpr int kSpread = 18;
// The same of two dimensions of V, by each one's largest value in the walk:
// what is dropped meets every key, and is 2^-25 of the dimension's scale at
// this ratio (error of the worst of 128 dimensions, fp32 steps / split, one of
// them 2^14 above the others 3.1e-7 / 2.9e-7, 2^16 3.1 / 5.0, 2^20 3.3 / 99).
constexpr int kSpreadCh = 14;
// The largest exponent of a query's largest value times a block's largest key
// value (log2 units). What the parts of a small q drop meets a large K and the
// reverse: 2^-39 of that product a dimension, so up to D / 2 * 2^-27 (2^-20 of
// a probability at dim 256) if large and small meet in every dimension and all
// roundings have one sign. Such a case at dim 256, error of the result on fp32
// steps / split: product 2^12 3e-8 / 2.7e-7, 2^14 6e-9 / 1.2e-6.
constexpr int kScoreExp = 12;

template <int D, bool KPOS>
__global__ __launch_bounds__(64 * SplitCfg<D>::NW)
__attribute__((amdgpu_waves_per_eu(D == 256 ? 1 : 2))) void attn_split_kernel(AttnParams p) {
    using C = SplitCfg<D>;
    constexpr int NT = D / 32, NS = D / 16;
    __shared__ __attribute__((aligned(16))) _Float16 smem[2][C::BUF];
    __shared__ float s_kf[2][C::NW];   // 2^(e - 14) of each wave's keys
    __shared__ int s_ev[2][C::NW];     // exponent of each wave's values
    __shared__ int s_bad[2];           // operands that the split would not carry (by buffer)
    __shared__ int s_redo;             // sums that are not finite, or not precise
    __shared__ int s_eq;               // the largest query exponent
    __shared__ int s_er[2][C::NW];     // each wave's value exponents: smallest, largest
    __shared__ uint32_t s_ch[D];       // the largest |value| of each dimension (its bits)
    __shared__ int32_t s_kp[2][C::KT];
    __shared__ int32_t s_q[2][4];
    __shared__ float s_qe[kSplitVecs];   // 2^(e - 14) of each query

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int qg = wave & 3, gk = wave >> 2;
    const int n = lane & 31, h = lane >> 5;
    const int kh = blockIdx.y;
    const uint32_t n_vec = (uint32_t)p.n_q * (uint32_t)p.rep;
    const uint32_t tile = gridDim.z - 1 - blockIdx.z;
    const int n_kv = (int)p.n_kv;

    // the lane's query vector: token tq, head kh * rep + u % rep
    const uint32_t u = tile * kSplitVecs + qg * 32 + n;
    const bool qok = u < n_vec;
    const uint32_t uc = qok ? u : n_vec - 1;
    const uint32_t tq = uc / (uint32_t)p.rep;
    const uint32_t qrow = tq * (uint32_t)p.n_head + (uint32_t)(kh * p.rep) + uc % (uint32_t)p.rep;
    const int32_t qp = p.qpos ? p.qpos[tq] : (int32_t)tq;

    // The wave's share of its group's queries (32 / GK rows, whole rows at a
    // time), loaded before the positions are known.
    constexpr int LQ = D / 4, PQ = 64 / LQ, NQ = 32 / C::GK / PQ;
    const int r0 = gk * (32 / C::GK) + lane / LQ, lq = lane % LQ;
    v4f f[NQ];
#pragma unroll
    for (int x = 0; x < NQ; ++x) {
        const uint32_t row = (uint32_t)__shfl((int)qrow, r0 + PQ * x);
        f[x] = *reinterpret_cast<const v4f*>(p.q + (int64_t)row * D + 4 * lq);
    }

    int32_t qmin = qp, qmax = qp;
#pragma unroll
    for (int off = 16; off >= 1; off >>= 1) {
        qmin = min(qmin, __shfl_xor(qmin, off));
        qmax = max(qmax, __shfl_xor(qmax, off));
    }
    qmin = __builtin_amdgcn_readfirstlane(qmin);
    qmax = __builtin_amdgcn_readfirstlane(qmax);
    for (int d = threadIdx.x; d < D; d += 64 * C::NW) s_ch[d] = 0;
    if (lane == 0 && gk == 0) {
        s_q[0][qg] = qmin;
        s_q[1][qg] = qmax;
        if (qg == 0) {
            s_bad[0] = s_bad[1] = s_redo = 0;
            s_eq = -1000;
        }
    }
    __syncthreads();
    const int32_t wmin = __builtin_amdgcn_readfirstlane(
        min(min(s_q[0][0], s_q[0][1]), min(s_q[0][2], s_q[0][3])));
    const int32_t wmax = __builtin_amdgcn_readfirstlane(
        max(max(s_q[1][0], s_q[1][1]), max(s_q[1][2], s_q[1][3])));

    // key tiles [i_lo, i_hi) that can hold kept keys (as attn_mfma_kernel)
    int i_lo = 0, i_hi = (n_kv + C::KT - 1) / C::KT;
    if constexpr (!KPOS) {
        i_hi = (int)min<int64_t>(i_hi, max<int64_t>(0, ((int64_t)wmax + C::KT) / C::KT));
        if (p.window > 0)
            i_lo = (int)max<int64_t>(0, ((int64_t)wmin - p.window + 1) / C::KT);
    }

    // A tile on its way to LDS, through buffer descriptors of the tile (keys
    // at or past n_kv read as zeros): of a wave's KW keys, lane (lane / LK,
    // lane % LK) takes dimensions 4lk .. +3 and D/2 + 4lk .. +3 of key PK * pass
    // + lane / LK of K (adjacent in LDS, as in q's rows there: a dot product
    // does not depend on the order of its terms), and 2 dimensions of the 8 keys of one octet of V (octet o of a sub-tile: keys
    // 16(o / 2) + 4(o % 2) + r and 8 more, the order of its 16 bytes of V^T).
    const int lk = lane % C::LK, pk = lane / C::LK;
    const int vo = D == 64 ? wave * 2 + (lane >> 5) : wave;
    const int vd = D == 64 ? 2 * (lane & 31) : 2 * lane;
    const int vk = 32 * (vo >> 2) + 16 * ((vo >> 1) & 1) + 4 * (vo & 1);
    const uint32_t kstride = (uint32_t)(p.n_head_kv * D * 4);
    const uint32_t koff = (uint32_t)(wave * C::KW + pk) * kstride + (uint32_t)lk * 16u;
    const uint32_t voff = (uint32_t)vk * kstride + (uint32_t)vd * 4u;
    const uint8_t* kbase = reinterpret_cast<const uint8_t*>(static_cast<const float*>(p.k) +
                                                            (int64_t)kh * D);
    const uint8_t* vbase = reinterpret_cast<const uint8_t*>(static_cast<const float*>(p.v) +
                                                            (int64_t)kh * D);
    v4f kr[C::NK][2];
    v2f vr[C::CV][8];
    int32_t kpr = 0;
    // a descriptor of the keys from key0 on (its size: the tile at most)
    auto rsrc = [&](const uint8_t* base, int key0) __attribute__((always_inline)) {
        const int left = min(n_kv - key0, C::KT);
        return __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint8_t*>(base) + (int64_t)key0 * kstride, 0,
            left > 0 ? (int)((uint32_t)(left - 1) * kstride + D * 4) : 0, kBufferDword3);
    };
    // load x of a tile: 2 NK of K, 8 CV of V (a descriptor each: the lane's
    // offsets are the same for all, so no registers hold the others)
    constexpr int NL = 2 * C::NK + 8 * C::CV;
    auto load1 = [&](int i, int x) __attribute__((always_inline)) {
        if (x < 2 * C::NK) {
            kr[x >> 1][x & 1] = __builtin_bit_cast(
                v4f, __builtin_amdgcn_raw_buffer_load_b128(
                         rsrc(kbase, i * C::KT + (x >> 1) * C::PK), (int)(koff + 2u * D * (x & 1)),
                         0, 0));
        } else {
            const int e = (x - 2 * C::NK) & 7, c = (x - 2 * C::NK) >> 3;
            vr[c][e] = __builtin_bit_cast(
                v2f, __builtin_amdgcn_raw_buffer_load_b64(
                         rsrc(vbase, i * C::KT + (e >> 2) * 8 + (e & 3)), (int)(voff + 512u * c),
                         0, 0));
        }
        if constexpr (KPOS) {   // (lane's key of the wave's KW)
            if (x == 0)
                kpr = p.kpos[min(i * C::KT + wave * C::KW + (lane & (C::KW - 1)), n_kv - 1)];
        }
    };
    auto load = [&](int i) __attribute__((always_inline)) {
#pragma unroll
        for (int x = 0; x < NL; ++x) load1(i, x);
    };
    // the loaded tile (i), on its way to buffer b: keys that nothing keeps
    // zeroed, the scales
    float fk, fv;
    int ek_lim = 0, ev_lo = 1000, ev_hi = -1000;
    float vch[C::CV][2];   // the largest value of each of the lane's dimensions
#pragma unroll
    for (int x = 0; x < C::CV; ++x) vch[x][0] = vch[x][1] = 0.0f;
    auto scales = [&](int b, int i) __attribute__((always_inline)) {
        const int first = i * C::KT + wave * C::KW;
        // keys of the tile that no query of the workgroup keeps become zeros
        auto visible = [&](int key, int32_t kp) __attribute__((always_inline)) {
            return key < n_kv && kp <= wmax && (p.window <= 0 || (int64_t)wmin - kp < p.window);
        };
        if constexpr (KPOS) {
            if (lane < C::KW) s_kp[b][wave * C::KW + lane] = kpr;
        }
        if (KPOS || (i + 1) * C::KT - 1 > wmax ||
            (p.window > 0 && (int64_t)wmin - i * C::KT >= p.window)) {
            asm volatile("");
#pragma unroll
            for (int x = 0; x < C::NK; ++x) {
                const int key = first + x * C::PK + pk;
                int32_t kp = key;
                if constexpr (KPOS) kp = __shfl(kpr, x * C::PK + pk);
                const bool vis = visible(key, kp);
#pragma unroll
                for (int y = 0; y < 8; ++y)
                    kr[x][y >> 2][y & 3] = vis ? kr[x][y >> 2][y & 3] : 0.0f;
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int key = i * C::KT + vk + (e >> 2) * 8 + (e & 3);
                int32_t kp = key;
                if constexpr (KPOS) kp = p.kpos[min(key, n_kv - 1)];
                const bool vis = visible(key, kp);
#pragma unroll
                for (int x = 0; x < C::CV; ++x) {
                    vr[x][e].x = vis ? vr[x][e].x : 0.0f;
                    vr[x][e].y = vis ? vr[x][e].y : 0.0f;
                }
            }
        }
        float ak = 0.0f, av = 0.0f;
#pragma unroll
        for (int x = 0; x < C::NK; ++x)
#pragma unroll
            for (int y = 0; y < 8; y += 2)
                ak = max3_abs(ak, kr[x][y >> 2][y & 3], kr[x][y >> 2][(y & 3) + 1]);
        // (a dimension's largest first: the lane keeps the walk's)
#pragma unroll
        for (int x = 0; x < C::CV; ++x) {
            float c[2] = {0.0f, 0.0f};
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                c[0] = max3_abs(c[0], vr[x][e].x, vr[x][e + 1].x);
                c[1] = max3_abs(c[1], vr[x][e].y, vr[x][e + 1].y);
            }
            av = max3(av, c[0], c[1]);
            vch[x][0] = max3(vch[x][0], c[0], c[0]);
            vch[x][1] = max3(vch[x][1], c[1], c[1]);
        }
        wave_max2(ak, av);
        const int ek = block_exp(ak), ev = block_exp(av);
        if (ev > -112) {
            // The smallest of the rows (keys) of V that are not zeros. In most
            // blocks one lane (of each half at head dim 64) sees in its first
            // dimension that all are within 2^-5 of the largest; else (keys
            // that nothing keeps among them) the rows' own maxima.
            float mn = vr[0][0].x;
            mn = min3_abs(mn, vr[0][1].x, vr[0][2].x);
            mn = min3_abs(mn, vr[0][3].x, vr[0][4].x);
            mn = min3_abs(mn, vr[0][5].x, vr[0][6].x);
            mn = min3_abs(mn, vr[0][7].x, vr[0][7].x);
            const uint64_t near = __ballot(mn >= av * 0.03125f);
            int lo = ev - 5;
            if (D == 64 ? (uint32_t)near == 0 || (near >> 32) == 0 : near == 0) {
                asm volatile("");   // (a branch)
                float low = av;
#pragma unroll
                for (int e = 0; e < 8; e += 2) {
                    float r0 = 0.0f, r1 = 0.0f;
#pragma unroll
                    for (int x = 0; x < C::CV; ++x) {
                        r0 = max3_abs(r0, vr[x][e].x, vr[x][e].y);
                        r1 = max3_abs(r1, vr[x][e + 1].x, vr[x][e + 1].y);
                    }
                    if constexpr (D == 64) {
                        half_max2(r0, r1);
                        const float o0 = lane_value(r0, 31), o1 = lane_value(r1, 31);
                        low = fminf(low, o0 > 0.0f ? o0 : av);
                        low = fminf(low, o1 > 0.0f ? o1 : av);
                        r0 = lane_value(r0, 63);
                        r1 = lane_value(r1, 63);
                    } else {
                        wave_max2(r0, r1);
                    }
                    low = fminf(low, r0 > 0.0f ? r0 : av);
                    low = fminf(low, r1 > 0.0f ? r1 : av);
                }
                lo = __builtin_amdgcn_readfirstlane(block_exp(low));
            }
            ev_lo = min(ev_lo, lo);
            ev_hi = max(ev_hi, ev);
        }
        if (lane == 0) {
            s_kf[b][wave] = pow2i(ek - 14);
            s_ev[b][wave] = ev;
            if (ev > 128 || ek > ek_lim || ev_hi - ev_lo > kSpread) s_bad[b] = 1;
        }
        fk = pow2i(14 - ek);
        fv = pow2i(14 - ev);
    };
    // pair y (of 4) of piece x (8 elements) of the loaded tile's split; the
    // piece goes to buffer b with its last pair
    h2 chi[4], clo[4];
    auto convert = [&](int b, int x, int y) __attribute__((always_inline)) {
        _Float16* o;
        int part;
        if (x < C::NK) {
            split_pair(kr[x][y >> 1][2 * (y & 1)] * fk, kr[x][y >> 1][2 * (y & 1) + 1] * fk,
                       chi[y], clo[y]);
            o = smem[b] + (wave * C::KW + pk + x * C::PK) * C::KP + 8 * lk;
            part = C::KPART;
        } else {
            // V^T row (a dimension): the octet's 16 bytes, swizzled by the
            // dimension so that a column of rows covers the banks
            const int c = (x - C::NK) >> 1, d = (x - C::NK) & 1;
            split_pair(vr[c][2 * y][d] * fv, vr[c][2 * y + 1][d] * fv, chi[y], clo[y]);
            o = smem[b] + 2 * C::KPART + ((vo >> 2) * D + vd + 128 * c + d) * C::VP +
                ((vo & 3) ^ ((vd >> 4) & 3)) * 8;
            part = C::VPART;
        }
        if (y == 3) {
            *reinterpret_cast<uint4*>(o) =
                make_uint4(h2_u32(chi[0]), h2_u32(chi[1]), h2_u32(chi[2]), h2_u32(chi[3]));
            *reinterpret_cast<uint4*>(o + part) =
                make_uint4(h2_u32(clo[0]), h2_u32(clo[1]), h2_u32(clo[2]), h2_u32(clo[3]));
        }
    };

    if (i_lo < i_hi) load(i_lo);

    // the positions the lane's query keeps: klo .. qp (khi without key
    // positions, where the key's place bounds them too)
    const int32_t klo = p.window > 0 ? (int32_t)max<int64_t>((int64_t)qp - p.window + 1,
                                                             KPOS ? INT32_MIN : 0)
                                     : (KPOS ? INT32_MIN : 0);
    const int32_t klo_max =
        p.window > 0 ? (int32_t)max<int64_t>((int64_t)qmax - p.window + 1, 0) : 0;
    const int32_t khi = max(min(qp, n_kv - 1), -1);

    // the query's parts, times scale * log2(e) (its product with two floats,
    // so that the scores' factor c is a power of two), through LDS into the
    // matrix operand's order: dimensions 16st + 8h .. +7 of step st.
    h8 qhi[NS], qlo[NS];
    float qsc;
    {
        constexpr int QPART = kSplitVecs * C::KP;
        static_assert(4 * QPART <= (int)sizeof(smem), "query staging");
        _Float16* qs = &smem[0][0];
        const float c0 = p.scale * kLog2e;
        const float c1 = __builtin_fmaf(p.scale, kLog2e, -c0) + p.scale * kLog2eLo;
        float amax[NQ];
#pragma unroll
        for (int x = 0; x < NQ; ++x) amax[x] = max3_abs(max3_abs(0.0f, f[x][0], f[x][1]), f[x][2], f[x][3]);
#pragma unroll
        for (int x = 0; x < NQ; x += 2) {
            row_max2(amax[x], amax[x + 1]);
#pragma unroll
            for (int y = x; y < x + 2; ++y) {
                if constexpr (LQ >= 32) amax[y] = fmaxf(amax[y], __shfl_xor(amax[y], 16));
                if constexpr (LQ >= 64) amax[y] = fmaxf(amax[y], __shfl_xor(amax[y], 32));
            }
        }
#pragma unroll
        for (int x = 0; x < NQ; ++x) {
            const int eq = block_exp(amax[x] * fabsf(c0) * 1.0001f);
            const float f0 = pow2i(14 - eq);
            if (lq == 0) {
                s_qe[qg * 32 + r0 + PQ * x] = pow2i(eq - 14);
                if (eq > 128) s_bad[0] = 1;
                atomicMax(&s_eq, eq);
            }
            h2 hi[2], lo[2];
#pragma unroll
            for (int y = 0; y < 4; ++y)
                f[x][y] = __builtin_fmaf(f[x][y], c0, f[x][y] * c1) * f0;
            split_pair(f[x][0], f[x][1], hi[0], lo[0]);
            split_pair(f[x][2], f[x][3], hi[1], lo[1]);
            _Float16* o = qs + (qg * 32 + r0 + PQ * x) * C::KP + 8 * (lq % (LQ / 2)) +
                          4 * (lq / (LQ / 2));
            *reinterpret_cast<uint2*>(o) = make_uint2(h2_u32(hi[0]), h2_u32(hi[1]));
            *reinterpret_cast<uint2*>(o + QPART) = make_uint2(h2_u32(lo[0]), h2_u32(lo[1]));
        }
        __syncthreads();
        const _Float16* qf = qs + (qg * 32 + n) * C::KP + 8 * h;
#pragma unroll
        for (int st = 0; st < NS; ++st) {
            qhi[st] = *reinterpret_cast<const h8*>(qf + 16 * st);
            qlo[st] = *reinterpret_cast<const h8*>(qf + 16 * st + QPART);
        }
        qsc = s_qe[qg * 32 + n];
        ek_lim = __builtin_amdgcn_readfirstlane(min(kScoreExp - s_eq, 128));
        __syncthreads();
    }

    // reference max (log2 units, a whole number: it and the exponents add
    // exactly), sum of p
    int m = kNoMax;
    float ls = 0.0f;
    int e_acc = -112;                 // the sums' exponent E
    v16f acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int x = 0; x < 16; ++x) acc[t][x] = 0.0f;

    // sub-tile sub of tile i in buffer b; with CONV the loaded tile is split
    // into the other buffer between the scores' matrix steps, and the one
    // after it loaded
    auto compute = [&](auto conv, int b, int sub, int i) __attribute__((always_inline)) {
        constexpr bool CONV = decltype(conv)::value;
        const int kb = i * C::KT + 32 * sub;
        constexpr int PS = 4 * C::NP / NS;   // pairs split a step
        const _Float16* kl = smem[b] + (32 * sub + n) * C::KP + 8 * h;
        // (the small products in sums of their own: their roundings vanish,
        // and the large ones meet half as many)
        v16f s, sl;
#pragma unroll
        for (int x = 0; x < 16; ++x) s[x] = sl[x] = 0.0f;
        h8 kph[2], kpl[2];
        // (the matrix steps go before the other wave's vector instructions:
        // 2048 causal tokens at head dim 64 97.1 -> 93.7 us, at 256 151.7 ->
        // 148.4, at 128 162 -> 160 on MI355X)
        __builtin_amdgcn_s_setprio(1);
        kph[0] = *reinterpret_cast<const h8*>(kl);
        kpl[0] = *reinterpret_cast<const h8*>(kl + C::KPART);
#pragma unroll
        for (int st = 0; st < NS; ++st) {
            // the next step's keys are read ahead; between the matrix steps
            // run the split's instructions
            if (st + 1 < NS) {
                kph[(st + 1) & 1] = *reinterpret_cast<const h8*>(kl + 16 * (st + 1));
                kpl[(st + 1) & 1] = *reinterpret_cast<const h8*>(kl + 16 * (st + 1) + C::KPART);
            }
            __builtin_amdgcn_sched_barrier(0);
            sl = __builtin_amdgcn_mfma_f32_32x32x16_f16(kpl[st & 1], qhi[st], sl, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kph[st & 1], qhi[st], s, 0, 0, 0);
            sl = __builtin_amdgcn_mfma_f32_32x32x16_f16(kph[st & 1], qlo[st], sl, 0, 0, 0);
            if constexpr (CONV) {
#pragma unroll
                for (int x = 0; x < PS; ++x)
                    convert(b ^ 1, (st * PS + x) >> 2, (st * PS + x) & 3);
#pragma unroll
                for (int x = 0; x < 3; ++x) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, 2 * PS, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_s_setprio(0);
#pragma unroll
        for (int x = 0; x < 16; ++x) s[x] += sl[x];
        // elements 4j .. 4j+3: keys 8j + 4h + r
        float c[4];
        int evt = -1000;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            // (at least the smallest normal: -inf times c stays -inf)
            c[j] = fmaxf(s_kf[b][(32 * sub + 8 * j) / C::KW] * qsc, 1.17549435e-38f);
            evt = max(evt, __builtin_amdgcn_readfirstlane(s_ev[b][(4 * sub + j) / C::OW]));
        }
        if (KPOS || kb + 31 > min(qmin, n_kv - 1) || kb < klo_max) {
            asm volatile("");   // (a branch: most steps skip this)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int i = 8 * j + r;   // key kb + i + 4h
                    bool keep;
                    if constexpr (KPOS) {
                        const int32_t kp = s_kp[b][32 * sub + i + 4 * h];
                        keep = kp <= qp && kp >= klo && kb + i + 4 * h < n_kv;
                    } else {
                        keep = i <= khi - kb - 4 * h && i >= klo - kb - 4 * h;
                    }
                    s[4 * j + r] = keep ? s[4 * j + r] : -INFINITY;
                }
        }
        float tm = -INFINITY;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float a = max3(s[4 * j], s[4 * j + 1], s[4 * j + 2]);
            tm = max3(tm, a * c[j], s[4 * j + 3] * c[j]);
        }
        tm = fmaxf(tm, __shfl_xor(tm, 32));

        // the sums follow the values' exponent (down only past 2^8, and not to
        // a tile of zeros; sums that overflow for it are redone at the end)
        // and the running max
        const int e_new = evt > e_acc || (evt < e_acc - 8 && evt > -112) ? evt : e_acc;
        // (the ceiling as a whole number; nothing kept, or a NaN: no max)
        const int mt = tm > -INFINITY ? (int)ceilf(fminf(fmaxf(tm, -1e8f), 1e8f)) : kNoMax;
        const int mn = max(m, mt);
        const int da = max(m - mn, -1000) + e_acc - e_new;
        const float alpha = da < -126 ? 0.0f : (da > 127 ? INFINITY : pow2i(da));
        ls *= m - mn < -126 ? 0.0f : pow2i(m - mn);
        m = mn;
        e_acc = e_new;
        const float msafe = m == kNoMax ? 0.0f : (float)m;   // p = 0 for a masked key
        // p in units of 2^(ev - E), ev the octet's (keys 16k + 4h + r and 8
        // more: elements 8k .. 8k+7); times 2^14 apart, so that the exponents
        // that matter are near zero, where they round least
        h8 phi[2], plo[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int fe = max(s_ev[b][(4 * sub + 2 * k + h) / C::OW] - e_acc, -54);
            const float off = (float)fe - msafe;
            float ps[4];
            h2 hi[4], lo[4];
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                const float cj = c[2 * k + (x >> 1)];
                const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[8 * k + 2 * x], cj, off));
                const float p1 =
                    __builtin_amdgcn_exp2f(__builtin_fmaf(s[8 * k + 2 * x + 1], cj, off));
                ps[x] = p0 + p1;
                split_pair(p0 * 16384.0f, p1 * 16384.0f, hi[x], lo[x]);
            }
            ls += ((ps[0] + ps[1]) + (ps[2] + ps[3])) * pow2i(-fe);
            phi[k] = __builtin_bit_cast(h8, make_uint4(h2_u32(hi[0]), h2_u32(hi[1]),
                                                       h2_u32(hi[2]), h2_u32(hi[3])));
            plo[k] = __builtin_bit_cast(h8, make_uint4(h2_u32(lo[0]), h2_u32(lo[1]),
                                                       h2_u32(lo[2]), h2_u32(lo[3])));
        }
        const _Float16* vl = smem[b] + 2 * C::KPART + (sub * D + n) * C::VP;
        // A step's keys are summed from zero and added to the sums once. During
        // the matrix steps of 16 keys the next values are read, the last
        // product of 32 dimensions is added to the sums, and (with CONV) a
        // share of the next tile's loads is issued.
        auto value = [&](int y) __attribute__((always_inline)) {   // y = 2t + k
            return vl + 32 * (y >> 1) * C::VP + ((2 * (y & 1) + h) ^ ((2 * (y >> 1) + (n >> 4)) & 3)) * 8;
        };
        v16f o[2];
        h8 vph[2], vpl[2];
        __builtin_amdgcn_s_setprio(1);
        vph[0] = *reinterpret_cast<const h8*>(value(0));
        vpl[0] = *reinterpret_cast<const h8*>(value(0) + C::VPART);
#pragma unroll
        for (int y = 0; y < 2 * NT; ++y) {
            const int t = y >> 1, k = y & 1, q = t & 1;
            if (y + 1 < 2 * NT) {
                vph[k ^ 1] = *reinterpret_cast<const h8*>(value(y + 1));
                vpl[k ^ 1] = *reinterpret_cast<const h8*>(value(y + 1) + C::VPART);
            }
            if constexpr (CONV) {
#pragma unroll
                for (int x = 0; x < NL; ++x)
                    if (x * 2 * NT / NL == y) load1(i + 2, x);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (k == 0) {
#pragma unroll
                for (int x = 0; x < 16; ++x) o[q][x] = 0.0f;
            }
            o[q] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vpl[k], phi[k], o[q], 0, 0, 0);
            o[q] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vph[k], plo[k], o[q], 0, 0, 0);
            o[q] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vph[k], phi[k], o[q], 0, 0, 0);
            if (t > 0) {
#pragma unroll
                for (int x = 8 * k; x < 8 * k + 8; ++x)
                    acc[t - 1][x] = __builtin_fmaf(acc[t - 1][x], alpha, o[q ^ 1][x]);
#pragma unroll
                for (int x = 0; x < 3; ++x) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_s_setprio(0);
#pragma unroll
        for (int x = 0; x < 16; ++x)
            acc[NT - 1][x] = __builtin_fmaf(acc[NT - 1][x], alpha, o[(NT - 1) & 1][x]);
    };

    if (i_lo < i_hi) {
        scales(0, i_lo);
#pragma unroll
        for (int x = 0; x < 4 * C::NP; ++x) convert(0, x >> 2, x & 3);
        load(i_lo + 1);
    }
    __syncthreads();
    // (s_bad[b] is written before the barrier that ends the step of buffer
    // b ^ 1 and not again before the next one: every wave reads the same)
    bool redo = false;
    for (int i = i_lo; i < i_hi; ++i) {
        const int b = (i - i_lo) & 1;
        const int flag = s_bad[b];
        // (past the last tile: zeros, into a buffer that nothing reads)
        scales(b ^ 1, i + 1);
        redo = __builtin_amdgcn_readfirstlane(flag) != 0;
        if (redo) break;
        compute(std::true_type{}, b, gk, i);
#pragma unroll
        for (int sub = gk + C::GK; sub < C::SUBS; sub += C::GK)
            compute(std::false_type{}, b, sub, i);
        __syncthreads();
    }
    if (!redo) {
        if (lane == 0) {
            s_er[0][wave] = ev_lo;
            s_er[1][wave] = ev_hi;
        }
#pragma unroll
        for (int x = 0; x < 2 * C::CV; ++x)
            atomicMax(&s_ch[vd + 128 * (x >> 1) + (x & 1)],
                      __builtin_bit_cast(uint32_t, vch[x >> 1][x & 1]));
        if constexpr (C::GK == 1) __syncthreads();
        // back to natural units, the halves of a column added
        ls += __shfl_xor(ls, 32);
        const int back = e_acc - 28;
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int x = 0; x < 16; ++x) acc[t][x] = ldexpf(acc[t][x], back);
        if constexpr (C::GK == 2) {
            // the second set of waves hands its sums to the first through LDS
            float* xs = reinterpret_cast<float*>(&smem[0][0]) + qg * (64 * (16 * NT + 2)) + lane;
            static_assert(4 * 64 * (16 * NT + 2) * 4 <= (int)sizeof(smem), "merge buffer");
            if (gk == 1) {
                xs[0] = (float)m;
                xs[64] = ls;
#pragma unroll
                for (int t = 0; t < NT; ++t)
#pragma unroll
                    for (int x = 0; x < 16; ++x) xs[64 * (2 + 16 * t + x)] = acc[t][x];
            }
            __syncthreads();
            if (gk == 0) {
                const float m0 = (float)m, m1 = xs[0], l1 = xs[64];
                const float mt = fmaxf(m0, m1);
                const float w0 = __builtin_amdgcn_exp2f(m0 - mt);
                const float w1 = __builtin_amdgcn_exp2f(m1 - mt);
                ls = ls * w0 + l1 * w1;
                m = max(m, (int)m1);
#pragma unroll
                for (int t = 0; t < NT; ++t)
#pragma unroll
                    for (int x = 0; x < 16; ++x)
                        acc[t][x] = acc[t][x] * w0 + xs[64 * (2 + 16 * t + x)] * w1;
            }
        }
#pragma unroll
        for (int x = 0; x < C::NW; ++x) {
            ev_lo = min(ev_lo, s_er[0][x]);
            ev_hi = max(ev_hi, s_er[1][x]);
        }
        // (a dimension of V far below the others; one of zeros is exact)
        bool faint = false;
#pragma unroll
        for (int d = lane; d < D; d += 64) {
            const uint32_t c = s_ch[d];
            faint = faint || (c != 0 && ev_hi - block_exp(__builtin_bit_cast(float, c)) > kSpreadCh);
        }
        // (scores past the clamp of m can leave no sum)
        bool bad = faint || ev_hi - ev_lo > kSpread || !(ls <= 3.4028235e38f) ||
                   (ls == 0.0f && m != kNoMax);
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int x = 0; x < 16; ++x) bad = bad || !(fabsf(acc[t][x]) <= 3.4028235e38f);
        bad = __any(bad) && gk == 0;
        if (bad && lane == 0) s_redo = 1;
        __syncthreads();
        redo = __builtin_amdgcn_readfirstlane(s_redo) != 0;
        if (!redo && gk == 0 && qok) {
            const float inv = 1.0f / fmaxf(ls, 1e-30f);
            // (64 bits: n_q * n_head rows, up to 2^31 - 1, of D elements)
            float* o = p.out + (int64_t)qrow * D + 4 * h;
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    *reinterpret_cast<v4f*>(o + 32 * t + 8 * j) =
                        v4f{acc[t][4 * j] * inv, acc[t][4 * j + 1] * inv, acc[t][4 * j + 2] * inv,
                            acc[t][4 * j + 3] * inv};
        }
    }
    if (redo) {
        TileSums<D>* sums = reinterpret_cast<TileSums<D>*>(&smem[0][0]);
        static_assert(C::GK * sizeof(TileSums<D>) <= sizeof(smem), "sums of the fp32 tiles");
#pragma unroll 1
        for (int x = gk; x < kSplitVecs / 16; x += C::GK) {
            __syncthreads();
            attn_tile_fp32<D>(p, (int64_t)tile * (kSplitVecs / 16) + x, kh, sums[gk]);
        }
    }
}
