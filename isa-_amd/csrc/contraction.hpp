// The projection as a contraction on the matrix cores (included by ekv_lut.hip).
//
// A branch current depends on x - w alone, and the thresholds of a layer lie in an interval
// [w_lo, w_hi] that is narrow against the width 2 n U_T over which the current changes. On it
//     f(x - w) = sum_j c_j(x) T_j(t),   t = (w - w_c) / w_h in [-1, 1],
// with Chebyshev polynomials T_j converges geometrically, whatever x is: the current's nearest
// singularities lie at (x - w) / (2 n U_T) = +-i pi, so the terms fall like rho^-j with
// rho = z + sqrt(z^2 + 1), z = pi * 2 n U_T / w_h (Trefethen, Approximation Theory and
// Approximation Practice, ch. 8). Both sums over cells become products of matrices whose inner
// index is (input, j):
//     Idiff[m, o]  = sum_(k, j) (c_j r)[m, k] (T_j(t+) - T_j(t-))[o, k]
//     dX[m, k]     = sum_j g_j(x[m, k]) H_j[m, k],  H_j = sum_o G[m, o] (T_j(t+) - T_j(t-))[o, k]
//     dVth+-[o, k] = -+ sum_j T_j(t+-[o, k]) S_j,   S_j = sum_m G[m, o] (d_j r)[m, k]
// with f' = sum_j d_j T_j and g_j = r (d_j - (r / V_sat) c_j): j = 0 cancels in the difference
// of the branches. R terms cost R products per cell and direction where the cell itself costs
// 32 (forward) or 52 (backward) VALU instructions, four or eight of them transcendental.
//
// Precision. Operands are kept to 22 bits as the sum of two f16 (hi + lo, scaled by a power of
// two per row so that the row's largest value is near 2^12), and every product is formed as
// hi hi + hi lo + lo hi in fp32 accumulators. The upper half of the terms is below 1e-3 of the
// lower half (their coefficients fall like rho^-j; for the slope's own sum, dVth, 4e-3) and is
// kept as single f16, 1e-7 of the result: 2 R products per cell instead of 3 R. (The formula's
// dVth keeps all its terms as pairs: its error before was 3.5e-7.) The differences
// T_j(t+) - T_j(t-) are formed in fp64 before they are rounded, so that a cell no longer loses the bits in which its two
// branches agree. c_j, d_j and g_j come from tables over x built per call in fp64 (cubic
// interpolation, step at most kSepStep of 2 n U_T: 2e-8 relative; the step is a power of two,
// so that a position within a step is exact in fp32).
//
// Measured (GPT-L layer 768 x 3072 at 2048 tokens, initial thresholds, R = 8): forward 4.30 ms
// by the per-cell kernels, 0.30 ms here; backward 8.17 and 0.74 ms; error against float64 of
// the forward 2.8e-6 and 2.6e-7, of dX 2.3e-6 and 3.4e-7, of dVth 3.5e-7 and 2.7e-7 (2-norm).
//
// Tables. A lookup is the line between two entries, L(c) = F(c) + S(c) a (1 - a) / 2 with F the
// smooth function through the entries, S its second difference and a the coordinate's fraction
// (the next term is smaller by the relative change from entry to entry, 1.5% at 4096 entries).
// With a (1 - a) = 1/6 - sum_q cos(2 pi q a) / (pi q)^2 and c = xs - ws,
//     L(xs - ws) = (F + S / 12)(xs - ws)
//                  - sum_q S(xs - ws) (cos 2 pi q xs cos 2 pi q ws + sin 2 pi q xs sin 2 pi q ws) / (2 pi^2 q^2):
// the first part is smooth and expands as above, the others are 1e-5 of it and take R / 4 terms
// of S per cosine and sine in plain f16. One harmonic keeps the forward's and dVth's remainder
// below the per-cell kernels' own rounding of coordinates and of the records' intercepts up to
// growths of 3.3% from entry to entry (about 3900 entries), and dX's, which they round less, up to
// 2.2% (about 6000); coarser tables take two, finer ones than about 14000 entries none. 2-norm
// against float64 lookups, initial thresholds, per-cell kernels against this: 4096 entries forward
// 9.8e-6 and 3.8e-6, dX 5.4e-6 and 3.2e-6, dVth 1.1e-6 and 8.1e-7; 5500 entries 9.1e-6 and 2.1e-6,
// 5.2e-6 and 1.7e-6, 1.2e-6 and 4.8e-7; 8192 entries 7.8e-6 and 9.9e-7, 5.6e-6 and 1.5e-6, 1.3e-6
// and 2.9e-7 (over 0.5 and 1 V also smaller, closest for
// dVth over 1 V at 4096 entries, 1.7e-6 and 1.6e-6). With two harmonics throughout 768 -> 3072
// at 8192 tokens took 1.06 ms forward and 2.47 backward, with one 0.92 and 2.35. Sums of T's
// differences give back the entries exactly. A table that is not smooth (bf16 entries) runs the
// per-cell kernels.
//
// R is chosen per call on the device from the thresholds' spread (sep_terms); a call whose
// operands do not suit (non-finite values, x near -V_sat or spread over more than the table
// holds, thresholds spread too far) runs the per-cell kernels, which return at once otherwise.

typedef _Float16 sep_h8 __attribute__((ext_vector_type(8)));
typedef _Float16 sep_h4 __attribute__((ext_vector_type(4)));
typedef _Float16 sep_h2 __attribute__((ext_vector_type(2)));
typedef float sep_f16 __attribute__((ext_vector_type(16)));
typedef unsigned sep_u4 __attribute__((ext_vector_type(4)));

constexpr int kSepStatX = 1024, kSepStatW = 256;  // blocks of the ranges of x and of the thresholds
constexpr int kSepStatG = 512;          // blocks of the largest |G| of each row
constexpr int kSepColChunks = 64;       // row chunks of a column pass, at most
constexpr int kSepGridMax = 16384;      // x-table points, at most
constexpr double kSepStep = 0.0148;     // x-table step in units of 2 n U_T
constexpr int kSepMaxTerms = 16;
constexpr int kSepLutMin = 2900, kSepLutMax = 65536;  // table entries: the kinks small enough, a thread per partial
constexpr float kSepQScale = 256.0f;    // of the threshold-side operand (values in [-2, 2])

// Widest threshold spread, in units of 2 n U_T, that R = 8 and 16 terms take: there the
// truncation is 1e-7 of the gradients (the forward's is ten times smaller). More would converge
// (16 terms to 4.4), but as the spread grows the per-cell kernels lose fewer bits to the branches'
// difference while the sums here have more terms: 2-norm against float64, 768 x 768 at 1900
// tokens, per-cell kernels against this, forward and dVth: 0.2142 V 2.8e-6 and 2.1e-7, 3.6e-7 and
// 2.5e-7; 0.3 V (1.4 units) 8.2e-7 and 3.7e-7, 3.0e-7 and 3.0e-7; 0.9 V 4.2e-7 and 4.2e-7, 3.1e-7
// and 3.3e-7. The formula goes over to the per-cell kernels where dVth's errors meet.
__host__ __device__ inline int sep_terms(float spread_u) { return spread_u <= 1.12f ? 8 : spread_u <= 1.45f ? 16 : 0; }

// Table calls: the lookups round more (over 1 V, 4.7 units, forward 2.7e-6 and 1.8e-6, dVth 1.7e-6
// and 1.6e-6 at 4096 entries), and 32 terms would cost what the lookups do.
__host__ __device__ inline int sep_terms_lut(float spread_u) { return spread_u <= 1.12f ? 8 : spread_u <= 5.0f ? 16 : 0; }

// What the passes of a call share, in its workspace.
struct SepHead {
    int terms;    // 0: the per-cell kernels run
    unsigned gmax;  // backward: bits of the largest |G|: not finite: the per-cell kernels run
    int rough;    // 1: the series does not converge as its terms assume, 2: a sample of the thresholds or of
                  // the table ruled the contraction out (then the other fields are not set): the per-cell kernels run
    int harmonics, harmonics_dx;  // of the table's kinks that are summed (0 to 2): forward and dVth, dX
    int n_grid;
    float xlo, xhi, wlo, whi;
    float lut_min, lut_scale;  // table coordinate (v - lut_min) * lut_scale
    float x0, step, inv_step; // table point i stands for x0 + i * step; step a power of two, x0 a multiple of it
    double wc, inv_wh, wh;   // t = (w - wc) * inv_wh
};

__device__ bool sep_takes(const SepHead* head) {
    return head != nullptr && __builtin_amdgcn_readfirstlane(head->terms != 0 && head->rough == 0 &&
                                                             head->gmax < 0x7f800000u) != 0;
}

struct SepArgs {
    const float* x;
    const float* wp;
    const float* wn;
    const float* g;          // backward: [M][ldg]
    int64_t M, K, O, ldg;
    const float* in_affine;
    float in_lo, in_hi;
    // formula
    double a, v_d;           // 1 / (2 n U_T), V_D
    double v_sat;
    int max_terms;
    // table (lut_n > 0): records {A, dT} or {A_I, dI, A_D, dD}
    const float* lut;
    int lut_n;
    double lut_min, lut_scale;
    double2* lut_val;        // [lut_n]: smooth part, second difference
    float2* lut_info;        // per 256 entries {largest relative growth from entry to entry, 1 where they do not suit}
    float* tabE;             // second difference's coefficients, -r e_i / (2 pi^2): [n_grid][R / 4]
    // workspace
    SepHead* head;
    float2* xpart;           // [kSepStatX]
    float2* wpart;           // [kSepStatW]
    float2* xrow;            // forward: [M] row ranges of x
    float2* xcol;            // backward: [kSepColChunks][K]
    unsigned* grow;          // backward: [M] largest |G| of a row (bits)
    unsigned* gcol;          // backward: [kSepColChunks][O]
    float* tab;              // forward c_j r (j = 1..R), backward d_j r (j = 0..R-1): [n_grid][R]
    float* tab2;             // backward g_j (j = 1..R)
    _Float16* xop;           // forward [M][Kd], backward (pairs, lower terms) [rows][Md]
    _Float16* wop;           // forward [O][Kd], backward [rows][Od]
    _Float16* xops;          // backward, upper terms, singles: [rows][Md]
    _Float16* wops;          // [rows][Od]
    _Float16* xoph;          // backward, harmonics, singles: [rows][Md]
    _Float16* woph;          // [rows][Od]
    _Float16* gop;           // backward, pairs: [M][Od]
    _Float16* gopT;          // [O][Md]
    _Float16* goph;          // backward, singles: [M][Od]
    _Float16* gophT;         // [O][Md]
    float* xscale;           // forward [M], backward [K]: inverse scale of xop's rows
    float* gscale;           // backward [M]
    float* gscaleT;          // backward [O]
    float2* tT;              // backward [K][Op]: {t+, t-}
    int64_t Op;
    int need_x, need_w;
};

__device__ inline float sep_input(const SepArgs& a, float x, float s, float b) {
    return a.in_affine ? input_map(x, s, b, a.in_lo, a.in_hi) : x;
}

// Layouts. An operand's row is a run of slabs of 128 bytes: 32 inner elements as pairs (their hi
// halves, then their lo halves) or 64 single f16.
// Forward, a row's inner elements: the lower terms as pairs, ordered (j / 4, k, j % 4), the
// upper ones as singles likewise, then (tables) the harmonics as singles; inputs padded to 16.
// Backward, tokens or outputs inside, rows in blocks of eight: four terms of an even input and of
// the odd one after it, so that a lane of the matrix cores' result holds one input's. The lower
// terms, the upper ones and the harmonics are operands of their own.
// Harmonics: an input has R values in blocks of four, at 8 terms of each harmonic its two cosines
// and two sines, at 16 the first one's four cosines, its four sines, then the second one's.
__host__ __device__ inline int64_t sep_inputs(int64_t K) { return (K + 15) / 16 * 16; }
__host__ __device__ inline int64_t sep_slabs_pairs(int64_t K, int terms) { return sep_inputs(K) * (terms / 2) / 32; }
__host__ __device__ inline int64_t sep_slabs_singles(int64_t K, int terms, int harmonics) {
    return sep_inputs(K) * (terms / 2 + harmonics * terms / 2) / 64;
}
__host__ __device__ inline int64_t sep_slabs(int64_t n) { return (n + 31) / 32; }
__host__ __device__ inline int64_t sep_slabs64(int64_t n) { return (n + 63) / 64; }
// Row of input k's value v (of its `per`) among the backward's rows.
__host__ __device__ inline int64_t sep_row(int64_t k, int per, int v) {
    return ((k >> 1) * (per / 4) + (v >> 2)) * 8 + (k & 1) * 4 + (v & 3);
}

// ----------------------------------------------------------------------------------
// Statistics: ranges of x (per row forward, per column backward), of the thresholds, and the
// largest |G| of each row and column. NaN makes a range infinite and a maximum non-finite.
// HBM-bound: x, the thresholds and G are read once (G and, with both gradients, twice).
// ----------------------------------------------------------------------------------

__device__ inline void sep_minmax(float v, float& lo, float& hi) {
    const bool bad = v != v;
    lo = fminf(lo, bad ? -INFINITY : v);
    hi = fmaxf(hi, bad ? INFINITY : v);
}

__device__ inline void sep_wave_minmax(float& lo, float& hi) {
    for (int d = 32; d > 0; d >>= 1) {
        lo = fminf(lo, __shfl_xor(lo, d));
        hi = fmaxf(hi, __shfl_xor(hi, d));
    }
}

// Block b of the table's 256-entry ranges: its entries from the records' differences (each block
// sums those before its range itself), as the smooth part F + S / 12 and S, and whether they
// suit: fourth differences within 3e-6 of the entries (what the cubic interpolation and the two
// terms of the lookup's line leave out), and for the backward a slope table that is the current
// table's slope (dX takes the currents from it; within 2e-5 of the difference).
__device__ inline void sep_lut_block(const SepArgs& a, int b) {
    constexpr int kHalo = 2, kSpan = 256 + 2 * kHalo;
    __shared__ double s_t[kSpan];
    __shared__ double s_sum[4];
    __shared__ float s_growth[4];
    __shared__ int s_bad;
    const int t = threadIdx.x, n = a.lut_n;
    const bool bwd = a.tab2 != nullptr;
    const int rec = bwd ? 4 : 2, val = bwd ? 2 : 0;  // the slope table backward, the currents forward
    const float* r0 = a.lut + (size_t)kPad * rec;
    const int base = b * 256, first = max(base - kHalo, 0), count = min(n - first, kSpan);
    if (t == 0) s_bad = 0;
    double sum = 0.0;
    for (int j = t; j < first; j += 256) sum += (double)r0[(size_t)j * rec + val + 1];
    for (int d = 32; d > 0; d >>= 1) sum += __shfl_xor(sum, d);
    if ((t & 63) == 0) s_sum[t >> 6] = sum;
    for (int i = t; i < kSpan; i += 256)  // element i + 1 gets entry i's difference
        if (i + 1 < kSpan) s_t[i + 1] = i + 1 < count ? (double)r0[(size_t)(first + i) * rec + val + 1] : 0.0;
    __syncthreads();
    if (t == 0) s_t[0] = (double)a.lut[val] + ((s_sum[0] + s_sum[1]) + (s_sum[2] + s_sum[3]));  // entry 0, padded
    __syncthreads();
    for (int d = 1; d < kSpan; d <<= 1) {
        const double u = t >= d ? s_t[t - d] : 0.0;
        const double v = t < kSpan - 256 && t + 256 >= d ? s_t[t + 256 - d] : 0.0;
        __syncthreads();
        s_t[t] += u;
        if (t < kSpan - 256) s_t[t + 256] += v;
        __syncthreads();
    }
    const int j = base + t, i = j - first;
    float growth = 0.0f;
    bool bad = false;
    double second = 0.0;
    if (j >= 1 && j + 1 < n) second = s_t[i - 1] - 2.0 * s_t[i] + s_t[i + 1];
    if (j >= kHalo && j + kHalo < n) {
        const double m2 = s_t[i - 2], m1 = s_t[i - 1], v = s_t[i], p1 = s_t[i + 1], p2 = s_t[i + 2];
        const double fourth = fabs((m2 + p2) - 4.0 * (m1 + p1) + 6.0 * v);
        if (!(fourth <= 3e-6 * fabs(v) + 1e-42)) bad = true;
        if (v > 1e-30) growth = (float)((p1 - v) / v);
        if (bwd) {  // the current's difference against the slope's integral (error of fourth order)
            const double di = (double)r0[(size_t)j * 4 + 1];
            const double want = (0.5 * (v + p1) - ((p2 - p1) - (v - m1)) / 24.0) / a.lut_scale;
            const double cur = fabs((double)r0[(size_t)j * 4] + (double)(j + kPad) * di);
            if (!(fabs(di - want) <= 2e-5 * fabs(want) + 4e-7 * cur + 1e-42)) bad = true;
        }
    }
    if (j < n) a.lut_val[j] = make_double2(s_t[i] + second / 12.0, second);
    if (bad) atomicOr(&s_bad, 1);
    for (int d = 32; d > 0; d >>= 1) growth = fmaxf(growth, __shfl_xor(growth, d));
    if ((t & 63) == 0) s_growth[t >> 6] = growth;
    __syncthreads();
    if (t == 0)
        a.lut_info[b] = make_float2(fmaxf(fmaxf(s_growth[0], s_growth[1]), fmaxf(s_growth[2], s_growth[3])), (float)s_bad);
}

__device__ inline unsigned sep_bits(float v) { return __float_as_uint(v) & 0x7fffffffu; }

// Whether a sample of the operands already rules the contraction out: 128 thresholds spread wider
// than its terms reach, or 16 places of the table not smooth (entries rounded to bf16). Wave-uniform
// and the same in every wave of the launch. What the sample passes the full statistics judge; what
// it fails they would refuse too (a sample's spread, growth and roughness are at most the whole's).
// Four neighbours at each of 16 places: every wave of the launch reads them, and 64 places cost
// the launch 6 us of L2 requests.
__device__ inline bool sep_sample_refuses(const SepArgs& a) {
    const int lane = threadIdx.x & 63, place = lane >> 2, off = lane & 3;
    const uint64_t n = (uint64_t)(a.O * a.K);
    float lo = INFINITY, hi = -INFINITY;
    // scattered, so that they are not a few inputs' (n >= 128)
    const uint64_t f = (((((uint64_t)place * 0x9e3779b97f4a7c15u) >> 32) * (n - 3)) >> 32) + off;
    const float wp = a.wp[f], wn = a.wn[f];
    double ua = a.a;
    bool bad = false;
    if (a.lut_n > 0) {
        const bool bwd = a.tab2 != nullptr;  // entries {A, dT}, backward the slope table's
        const int i = 2 + (int)((int64_t)place * (a.lut_n - 6) / 16);
        const float2 r = *reinterpret_cast<const float2*>(a.lut + (size_t)(kPad + i - 2 + off) * (bwd ? 4 : 2) + (bwd ? 2 : 0));
        const double d0 = __shfl(r.y, place * 4), d1 = __shfl(r.y, place * 4 + 1), d2 = __shfl(r.y, place * 4 + 2),
                     d3 = __shfl(r.y, place * 4 + 3);
        const double v = (double)__shfl(r.x, place * 4 + 2) + (double)(i + kPad) * d2;  // entry i, to 1e-5
        bad = !(fabs((d3 - d0) - 3.0 * (d2 - d1)) <= 4e-6 * fabs(v) + 2e-42);
        float growth = v > 1e-30 ? (float)(d2 / v) : 0.0f;
        for (int d = 32; d > 0; d >>= 1) growth = fmaxf(growth, __shfl_xor(growth, d));
        ua = 0.5 * 0.999 * (double)growth * a.lut_scale;
    }
    sep_minmax(wp, lo, hi);
    sep_minmax(wn, lo, hi);
    sep_wave_minmax(lo, hi);
    const float spread = (float)(((double)hi - (double)lo) * ua);
    const int terms = a.lut_n > 0 ? sep_terms_lut(spread) : sep_terms(spread);
    return __builtin_amdgcn_readfirstlane((int)(__any(bad) || terms == 0 || terms > a.max_terms)) != 0;
}

// Blocks: kSepStatX of x, kSepStatW of the thresholds, (xcol) kSepColChunks x ceil(K / 256) of
// x's columns, ceil(lut_n / 256) of the table, then the layer glue's gradient blocks (glue.geff).
__global__ __launch_bounds__(256) void sep_stat_kernel(SepArgs a, PrepArgs prep, GlueGradArgs glue) {
    int b = blockIdx.x;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const float as = a.in_affine ? a.in_affine[0] : 1.0f, ab = a.in_affine ? a.in_affine[1] : 0.0f;
    const int lut_blocks = (a.lut_n + 255) / 256;
    const int xcols = a.xcol ? kSepColChunks * (int)((a.K + 255) / 256) : 0;
    if (b < kSepStatX + kSepStatW + lut_blocks + xcols) {
        const bool refuses = sep_sample_refuses(a);
        if (b == 0 && t == 0) {
            a.head->gmax = 0;
            a.head->rough = refuses ? 2 : 0;
            a.head->terms = 0;
        }
        if (refuses) {  // the per-cell kernels' prep at once, beside the glue's gradient
            static_assert(kSepStatX + kSepStatW == kPrepBlocksX + kPrepBlocksW, "the prep's blocks");
            if (b < kPrepBlocksX + kPrepBlocksW) prep_block(prep, b);
            return;
        }
    }
    if (b < kSepStatX) {
        float lo = INFINITY, hi = -INFINITY;
        if (a.xrow) {  // a wave per row
            for (int64_t m = (int64_t)b * 4 + wave; m < a.M; m += (int64_t)kSepStatX * 4) {
                float l = INFINITY, h = -INFINITY;
                const float* row = a.x + m * a.K;
                for (int64_t k = lane; k < a.K; k += 256) {
                    float v[4];
#pragma unroll
                    for (int q = 0; q < 4; ++q) v[q] = row[k + q * 64 < a.K ? k + q * 64 : k];
#pragma unroll
                    for (int q = 0; q < 4; ++q) sep_minmax(sep_input(a, v[q], as, ab), l, h);
                }
                sep_wave_minmax(l, h);
                if (lane == 0) a.xrow[m] = make_float2(l, h);
                lo = fminf(lo, l);
                hi = fmaxf(hi, h);
            }
        } else {
            const int64_t n = a.M * a.K, stride = (int64_t)kSepStatX * 256;
            for (int64_t e = (int64_t)b * 256 + t; e < n; e += 4 * stride) {
                float v[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) v[q] = a.x[e + q * stride < n ? e + q * stride : e];
#pragma unroll
                for (int q = 0; q < 4; ++q) sep_minmax(sep_input(a, v[q], as, ab), lo, hi);
            }
        }
        block_minmax(lo, hi, &a.xpart[b]);
        return;
    }
    b -= kSepStatX;
    if (b < kSepStatW) {
        float lo = INFINITY, hi = -INFINITY;
        const int64_t n = a.O * a.K, stride = (int64_t)kSepStatW * 256;
        for (int64_t e = (int64_t)b * 256 + t; e < n; e += 4 * stride) {
            float v[8];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int64_t f = e + q * stride < n ? e + q * stride : e;
                v[2 * q] = a.wp[f];
                v[2 * q + 1] = a.wn[f];
            }
#pragma unroll
            for (int q = 0; q < 8; ++q) sep_minmax(v[q], lo, hi);
        }
        block_minmax(lo, hi, &a.wpart[b]);
        return;
    }
    b -= kSepStatW;
    if (b < lut_blocks) {
        sep_lut_block(a, b);
        return;
    }
    b -= lut_blocks;
    if (b < xcols) {
        const int64_t rows = (a.M + kSepColChunks - 1) / kSepColChunks;
        const int chunk = b % kSepColChunks;
        const int64_t col = (int64_t)(b / kSepColChunks) * 256 + t;
        const int64_t m0 = chunk * rows, m1 = m0 + rows < a.M ? m0 + rows : a.M;
        if (col >= a.K) return;
        float lo = INFINITY, hi = -INFINITY;
#pragma unroll 8
        for (int64_t m = m0; m < m1; ++m) sep_minmax(sep_input(a, a.x[m * a.K + col], as, ab), lo, hi);
        a.xcol[(int64_t)chunk * a.K + col] = make_float2(lo, hi);
        return;
    }
    b -= xcols;
    glue_grad_block(glue, b % kGlueBlocks, b / kGlueBlocks, (int)(glue.Op / 256));
}

// The largest |G| of a row or column (blocks of the table kernel's launch).
__device__ inline void sep_grad_block(const SepArgs& a, int b) {
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    if (b < kSepStatG) {
        unsigned all = 0;
        for (int64_t m = (int64_t)b * 4 + wave; m < a.M; m += (int64_t)kSepStatG * 4) {
            unsigned h = 0;
            const float* row = a.g + m * a.ldg;
            for (int64_t o = lane; o < a.O; o += 256) {
                unsigned v[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) v[q] = sep_bits(row[o + q * 64 < a.O ? o + q * 64 : o]);
                h = max(h, max(max(v[0], v[1]), max(v[2], v[3])));
            }
            for (int d = 32; d > 0; d >>= 1) h = max(h, (unsigned)__shfl_xor((int)h, d));
            if (lane == 0) a.grow[m] = h;
            all = max(all, h);
        }
        __shared__ unsigned s_all;  // one atomic per block: they all meet at one address
        if (t == 0) s_all = 0;
        __syncthreads();
        if (lane == 0) atomicMax(&s_all, all);
        __syncthreads();
        if (t == 0) atomicMax(&a.head->gmax, s_all);
        return;
    }
    b -= kSepStatG;
    const int64_t rows = (a.M + kSepColChunks - 1) / kSepColChunks;
    const int chunk = b % kSepColChunks;
    const int64_t col = (int64_t)(b / kSepColChunks) * 256 + t;
    const int64_t m0 = chunk * rows, m1 = m0 + rows < a.M ? m0 + rows : a.M;
    if (col >= a.O) return;
    unsigned h = 0;
#pragma unroll 8
    for (int64_t m = m0; m < m1; ++m) h = max(h, sep_bits(a.g[m * a.ldg + col]));
    a.gcol[(int64_t)chunk * a.O + col] = h;
}

// ----------------------------------------------------------------------------------
// Mode and coefficient tables. Every block reduces the partials itself and block 0 records the
// result; a thread builds one table point: the slope at R Chebyshev points of the threshold
// interval, its coefficients d_j (Trefethen ch. 3: a discrete cosine sum), and c_j by
// integration, c_j = -(w_h / 2j) (d_(j-1) - d_(j+1)), which needs no difference of currents.
// ----------------------------------------------------------------------------------

__device__ inline double sep_slope(double v, double a, double v_d) {  // f'(v) of f = sp(u1)^2 - sp(u2)^2
    const double u1 = v * a, u2 = (v - v_d) * a;
    const double e1 = exp(-fabs(u1)), e2 = exp(-fabs(u2));
    const double s1 = log1p(e1) + fmax(u1, 0.0), s2 = log1p(e2) + fmax(u2, 0.0);
    const double g1 = (u1 >= 0.0 ? 1.0 : e1) / (1.0 + e1), g2 = (u2 >= 0.0 ? 1.0 : e2) / (1.0 + e2);
    return 2.0 * a * (s1 * g1 - s2 * g2);
}

// The lookup's smooth part (cubic) or its second difference (linear) at coordinate c, which
// lies two entries or more inside the table.
__device__ inline double sep_lut_smooth(const double2* val, int n, double c) {
    int i = (int)c;
    i = i < 1 ? 1 : i > n - 3 ? n - 3 : i;
    const double f = c - i, g = 1.0 - f;
    return -f * g * (1.0 + g) / 6.0 * val[i - 1].x + g * (1.0 + f) * (1.0 + g) * 0.5 * val[i].x +
           f * (1.0 + f) * (1.0 + g) * 0.5 * val[i + 1].x - f * g * (1.0 + f) / 6.0 * val[i + 2].x;
}

__device__ inline double sep_lut_second(const double2* val, int n, double c) {
    int i = (int)c;
    i = i < 1 ? 1 : i > n - 3 ? n - 3 : i;
    return val[i].y + (c - i) * (val[i + 1].y - val[i].y);
}

constexpr int kSepTableBlocks = 256;

// Blocks: kSepTableBlocks of the tables, then (g) kSepStatG of G's rows and kSepColChunks x
// ceil(O / 256) of its columns.
__global__ __launch_bounds__(256) void sep_table_kernel(SepArgs a) {
    __shared__ float2 s_x, s_w, s_info;
    __shared__ SepHead s_head;
    __shared__ double s_cos[4 * kSepMaxTerms], s_val[256], s_sec[256], s_d[256];
    const int t = threadIdx.x;
    const bool lut = a.lut_n > 0;
    // (other blocks of this launch set rough to 1, never to 2)
    if (__builtin_amdgcn_readfirstlane(a.head->rough) == 2) return;
    {
        float lo = INFINITY, hi = -INFINITY;
#pragma unroll
        for (int q = 0; q < kSepStatX / 256; ++q) {
            const float2 v = a.xpart[t + q * 256];
            lo = fminf(lo, v.x);
            hi = fmaxf(hi, v.y);
        }
        const float2 w = a.wpart[t];
        static_assert(kSepStatW == 256 && kSepLutMax <= 256 * 256, "a thread per partial");
        const float2 info = t * 256 < a.lut_n ? a.lut_info[t] : make_float2(0.0f, 0.0f);
        block_minmax(lo, hi, &s_x);
        __syncthreads();
        block_minmax(w.x, w.y, &s_w);
        __syncthreads();
        block_minmax(-info.y, info.x, &s_info);  // (-1 where some do not suit, growth)
        __syncthreads();
    }
    if (t == 0) {
        SepHead h{};
        const float xlo = s_x.x, xhi = s_x.y, wlo = s_w.x, whi = s_w.y;
        // a: the current's e-folds per volt of overdrive are 2 a at most
        const double growth = lut ? (double)s_info.y : 0.0;
        const double ua = lut ? 0.5 * growth * a.lut_scale : a.a;
        const double step = exp2(floor(log2(kSepStep / ua)));
        const double rlo = 1.0 + (double)xlo / a.v_sat, rhi = 1.0 + (double)xhi / a.v_sat;
        const double first = floor((double)xlo / step) - 1.0;
        const double points = floor((double)xhi / step) - first + 3.0;
        const bool finite = xlo > -1e30f && xhi < 1e30f && wlo > -1e30f && whi < 1e30f;
        const float spread = (float)(((double)whi - (double)wlo) * ua);
        const int terms = lut ? sep_terms_lut(spread) : sep_terms(spread);
        bool ok = finite && terms > 0 && terms <= a.max_terms && rlo > 0.1 && rhi > 0.1 &&
                  points <= (double)kSepGridMax && fmax(fabs((double)xlo), fabs((double)xhi)) < step * (1 << 23);
        if (lut) {  // every lookup inside the table, the x table's margin included
            h.harmonics = growth > 0.033 ? 2 : growth > 0.009 ? 1 : 0;
            h.harmonics_dx = growth > 0.022 ? 2 : h.harmonics;
            const double margin = 4.0 * step * a.lut_scale + 4.0;
            ok = ok && s_info.x == 0.0f && growth > 1e-6 && growth < 0.045 &&
                 ((double)xlo - (double)whi - a.lut_min) * a.lut_scale >= margin &&
                 ((double)xhi - (double)wlo - a.lut_min) * a.lut_scale <= (double)(a.lut_n - 1) - margin;
            h.lut_min = (float)a.lut_min;
            h.lut_scale = (float)a.lut_scale;
        } else {  // |u| far below the exponent range of fp64
            ok = ok && fmax(fabs((double)xlo), fabs((double)xhi)) * ua < 300.0 &&
                 fmax(fabs((double)wlo), fabs((double)whi)) * ua < 300.0;
        }
        if (ok) {
            h.terms = terms;
            h.n_grid = (int)points;
            h.x0 = (float)(first * step);
            h.step = (float)step;
            h.inv_step = (float)(1.0 / step);
            h.wc = 0.5 * ((double)wlo + (double)whi);
            h.wh = fmax(0.5 * ((double)whi - (double)wlo), 1e-3 / ua);
            h.inv_wh = 1.0 / h.wh;
        }
        h.xlo = xlo;
        h.xhi = xhi;
        h.wlo = wlo;
        h.whi = whi;
        s_head = h;
        if (blockIdx.x == 0) {  // all but gmax and rough, which other blocks add to
            SepHead* g = a.head;
            g->terms = h.terms;
            g->harmonics = h.harmonics;
            g->harmonics_dx = h.harmonics_dx;
            g->n_grid = h.n_grid;
            g->xlo = xlo;
            g->xhi = xhi;
            g->wlo = wlo;
            g->whi = whi;
            g->lut_min = h.lut_min;
            g->lut_scale = h.lut_scale;
            g->x0 = h.x0;
            g->step = h.step;
            g->inv_step = h.inv_step;
            g->wc = h.wc;
            g->inv_wh = h.inv_wh;
            g->wh = h.wh;
        }
    }
    __syncthreads();
    const SepHead h = s_head;
    const int R = h.terms;
    if (R == 0) return;
    if (blockIdx.x >= kSepTableBlocks) {
        sep_grad_block(a, blockIdx.x - kSepTableBlocks);
        return;
    }
    for (int q = t; q < 4 * R; q += 256) s_cos[q] = cospi((double)q / (2.0 * R));
    // a block takes 256 / R points at a time: a thread per (point, Chebyshev point), then per
    // (point, j)
    const int per = 256 / R, pl = t / R, n = t - pl * R;
    for (int i0 = blockIdx.x * per; i0 < h.n_grid; i0 += kSepTableBlocks * per) {
        const double x = (double)h.x0 + (double)(i0 + pl) * (double)h.step;
        const double r = 1.0 / (1.0 + x / a.v_sat);
        __syncthreads();
        const double v = x - (h.wc + h.wh * s_cos[2 * n + 1]);
        if (lut) {
            const double c = (v - a.lut_min) * a.lut_scale;
            s_val[t] = sep_lut_smooth(a.lut_val, a.lut_n, c);
            s_sec[t] = h.harmonics > 0 ? sep_lut_second(a.lut_val, a.lut_n, c) : 0.0;
        } else {
            s_val[t] = sep_slope(v, a.a, a.v_d);
        }
        __syncthreads();
        // the slope's d_n; the forward's tables hold currents: their coefficient n + 1 (of the
        // polynomial of degree R - 1, so that the last is zero)
        const int j = n + 1;
        const bool direct = lut && !a.tab2;
        const int jd = direct ? j : n;
        double d = 0.0;
        for (int q = 0; q < R; ++q) d += s_val[pl * R + q] * s_cos[(jd * (2 * q + 1)) % (4 * R)];
        d *= 2.0 / R;
        if (direct && j == R) d = 0.0;
        s_d[t] = d;
        double e2 = 0.0;
        if (h.harmonics > 0 && n < R / 4) {
            for (int q = 0; q < R; ++q) e2 += s_sec[pl * R + q] * s_cos[(n * (2 * q + 1)) % (4 * R)];
            e2 *= (n == 0 ? 1.0 : 2.0) / R;
        }
        __syncthreads();
        if (i0 + pl < h.n_grid) {
            const size_t e = (size_t)(i0 + pl) * R + n;
            if (direct) {
                a.tab[e] = (float)(d * r);
            } else {  // c_j from d_(j-1) = d and d_(j+1)
                const double d_next = j < R ? s_d[t + 1] : 0.0, d_after = j + 1 < R ? s_d[t + 2] : 0.0;
                const double c = -h.wh / (2.0 * j) * (d - d_after);
                if (a.tab2) {
                    a.tab[e] = (float)((n == 0 ? 0.5 * d : d) * r);
                    a.tab2[e] = (float)(r * (d_next - r / a.v_sat * c));
                } else {
                    a.tab[e] = (float)(c * r);
                }
            }
            if (h.harmonics > 0 && n < R / 4)
                a.tabE[(size_t)(i0 + pl) * (R / 4) + n] = (float)(-r * e2 * 0.050660591821168886);  // 1 / (2 pi^2)
            // the last coefficients of a table that grows otherwise than its steepest part says
            if (lut && n == 0) {
                const int last = direct ? R - 2 : R - 1;  // of degree R - 1
                double big = 0.0;
                for (int q = direct ? 0 : 1; q < R; ++q) big = fmax(big, fabs(s_d[t + q]));
                const double mean = direct ? 0.0 : fabs(0.5 * s_d[t]);
                if (!(fabs(s_d[t + last]) <= 2e-5 * big + 2e-6 * mean + 1e-35)) atomicOr(&a.head->rough, 1);
            }
        }
    }
}

// Position of x in a table: the first of its four points and their cubic weights.
struct SepAt {
    int i;
    float w[4];
};

__device__ inline SepAt sep_at(const SepHead& h, float x) {
    int i = (int)((x - h.x0) * h.inv_step);
    i = i < 1 ? 1 : i > h.n_grid - 3 ? h.n_grid - 3 : i;
    // x0 + i step is exact, and so is x's distance from it
    const float f = (x - (h.x0 + (float)i * h.step)) * h.inv_step, g = 1.0f - f;
    SepAt at;
    at.i = i - 1;
    at.w[0] = -f * g * (1.0f + g) * (1.0f / 6.0f);
    at.w[1] = g * (1.0f + f) * (1.0f + g) * 0.5f;
    at.w[2] = f * (1.0f + f) * (1.0f + g) * 0.5f;
    at.w[3] = -f * g * (1.0f + f) * (1.0f / 6.0f);
    return at;
}

__device__ inline float4 sep_eval4(const float* tab, int R, const SepAt& at, int j) {
    const float* p = tab + (size_t)at.i * R + j;
    const float4 v0 = *reinterpret_cast<const float4*>(p), v1 = *reinterpret_cast<const float4*>(p + R);
    const float4 v2 = *reinterpret_cast<const float4*>(p + 2 * R), v3 = *reinterpret_cast<const float4*>(p + 3 * R);
    float4 s;
    s.x = fmaf(at.w[3], v3.x, fmaf(at.w[2], v2.x, fmaf(at.w[1], v1.x, at.w[0] * v0.x)));
    s.y = fmaf(at.w[3], v3.y, fmaf(at.w[2], v2.y, fmaf(at.w[1], v1.y, at.w[0] * v0.y)));
    s.z = fmaf(at.w[3], v3.z, fmaf(at.w[2], v2.z, fmaf(at.w[1], v1.z, at.w[0] * v0.z)));
    s.w = fmaf(at.w[3], v3.w, fmaf(at.w[2], v2.w, fmaf(at.w[1], v1.w, at.w[0] * v0.w)));
    return s;
}

// The power of two that brings a largest value to [2^11, 2^12), and its inverse.
__device__ inline float sep_scale_of(float largest, float* inverse) {
    int e = 12;
    if (largest > 0.0f) e = 12 - (ilogbf(largest) + 1);
    e = e > 120 ? 120 : e < -120 ? -120 : e;
    *inverse = ldexpf(1.0f, -e);
    return ldexpf(1.0f, e);
}

// A row's largest |c_j r| or |d_j r|, from above: the first coefficient grows with x and
// dominates the others, r falls with x.
__device__ inline float sep_bound(const SepHead& h, const float* tab, int j, float2 range, float v_sat) {
    const SepAt at = sep_at(h, range.y);
    const float* p = tab + (size_t)at.i * h.terms + j;
    float s = 0.0f;
    for (int q = 0; q < 4; ++q) s = fmaf(at.w[q], p[q * h.terms], s);
    return fabsf(s) * (1.0f + range.y / v_sat) / (1.0f + range.x / v_sat) * 1.001f;
}

__device__ inline void sep_split(float v, _Float16& hi, _Float16& lo) {
    hi = (_Float16)v;
    lo = (_Float16)(v - (float)hi);
}

// Stores a pair of neighbouring inner elements (e, e + 1; e even) of a row of hi/lo slabs.
__device__ inline void sep_store2(_Float16* row, int64_t e, float v0, float v1) {
    sep_h2 hi, lo;
    _Float16 h0, l0, h1, l1;
    sep_split(v0, h0, l0);
    sep_split(v1, h1, l1);
    hi.x = h0; hi.y = h1; lo.x = l0; lo.y = l1;
    _Float16* p = row + (e >> 5) * 64 + (e & 31);
    *reinterpret_cast<sep_h2*>(p) = hi;
    *reinterpret_cast<sep_h2*>(p + 32) = lo;
}

// ----------------------------------------------------------------------------------
// Forward operands: xop[m] = c_j r (a wave per row, lanes along k) and wop[o] = T_j(t+) - T_j(t-),
// each (row, k) four values in 8-byte stores that neighbouring lanes continue. HBM-bound.
// ----------------------------------------------------------------------------------

constexpr int kSepExpandBlocks = 2048;

__device__ inline void sep_store4(_Float16* row, int64_t e, const float v[4]) {  // pairs
    sep_h4 hi, lo;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        _Float16 h, l;
        sep_split(v[q], h, l);
        hi[q] = h;
        lo[q] = l;
    }
    _Float16* p = row + (e >> 5) * 64 + (e & 31);
    *reinterpret_cast<sep_h4*>(p) = hi;
    *reinterpret_cast<sep_h4*>(p + 32) = lo;
}

__device__ inline void sep_store4h(_Float16* row, int64_t e, const float v[4]) {  // singles
    sep_h4 h;
#pragma unroll
    for (int q = 0; q < 4; ++q) h[q] = (_Float16)v[q];
    *reinterpret_cast<sep_h4*>(row + e) = h;
}

// Walks T_1, T_2, ... of both branches and hands out blocks of four differences.
struct SepChebPair {
    double p0 = 1.0, p1, n0 = 1.0, n1, tp, tn;
    __device__ SepChebPair(double a, double b) : p1(a), n1(b), tp(2.0 * a), tn(2.0 * b) {}
    __device__ void next4(float* v, float scale) {  // T_j(t+) - T_j(t-) of the next four j
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            v[q] = (float)(p1 - n1) * scale;
            const double p2 = tp * p1 - p0, n2 = tn * n1 - n0;
            p0 = p1;
            p1 = p2;
            n0 = n1;
            n1 = n2;
        }
    }
};

// cos and sin of 2 pi q theta, q = 1, 2 (theta in revolutions).
__device__ inline void sep_trig(float theta, float* c, float* sn) {
    const float f = theta - floorf(theta);
    c[0] = __builtin_amdgcn_cosf(f);
    sn[0] = __builtin_amdgcn_sinf(f);
    c[1] = 2.0f * c[0] * c[0] - 1.0f;
    sn[1] = 2.0f * sn[0] * c[0];
}

// Block blk of an input's harmonic values on the token side: the second difference's
// coefficients e times cosine and sine.
__device__ inline void sep_harm_x(float v[4], const float e[4], int terms, int blk, const float c[2], const float sn[2],
                                  float scale) {
    const float ca = c[0], cb = c[1], sa = sn[0], sb = sn[1];
    if (terms == 8) {
        const float f = blk ? 0.25f * scale : scale, fc = (blk ? cb : ca) * f, fs = (blk ? sb : sa) * f;
        v[0] = e[0] * fc;
        v[1] = e[1] * fc;
        v[2] = e[0] * fs;
        v[3] = e[1] * fs;
    } else {
        const float t = blk & 1 ? (blk & 2 ? sb : sa) : (blk & 2 ? cb : ca);
        const float f = t * (blk & 2 ? 0.25f * scale : scale);
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = e[i] * f;
    }
}

// Likewise on the threshold side: T_i(t+) cos - T_i(t-) cos, ...
__device__ inline void sep_harm_w(float v[4], const float tp[4], const float tn[4], int terms, int blk, const float cp[2],
                                  const float sp[2], const float cn[2], const float sn[2], float scale) {
    const float cpa = cp[0], cpb = cp[1], spa = sp[0], spb = sp[1], cna = cn[0], cnb = cn[1], sna = sn[0], snb = sn[1];
    if (terms == 8) {
        const float c0 = blk ? cpb : cpa, s0 = blk ? spb : spa, c1 = blk ? cnb : cna, s1 = blk ? snb : sna;
        v[0] = (c0 - c1) * scale;
        v[1] = (tp[1] * c0 - tn[1] * c1) * scale;
        v[2] = (s0 - s1) * scale;
        v[3] = (tp[1] * s0 - tn[1] * s1) * scale;
    } else {
        const float f0 = blk & 1 ? (blk & 2 ? spb : spa) : (blk & 2 ? cpb : cpa);
        const float f1 = blk & 1 ? (blk & 2 ? snb : sna) : (blk & 2 ? cnb : cna);
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = (tp[i] * f0 - tn[i] * f1) * scale;
    }
}

__device__ inline void sep_cheb4(float t, float v[4]) {  // T_0 .. T_3
    v[0] = 1.0f;
    v[1] = t;
    v[2] = 2.0f * t * t - 1.0f;
    v[3] = 2.0f * t * v[2] - t;
}

// The nearest table point's R / 4 second-difference coefficients (they change by 1.5% from
// point to point, and are 1e-5 of the result).
__device__ inline void sep_second(const SepHead& h, const float* tabE, const SepAt& at, float e[4]) {
    const size_t i = (size_t)(at.i + (at.w[2] > at.w[1] ? 2 : 1));
    if (h.terms == 8) {
        const float2 v = *reinterpret_cast<const float2*>(tabE + i * 2);
        e[0] = v.x; e[1] = v.y; e[2] = e[3] = 0.0f;
    } else {
        const float4 v = *reinterpret_cast<const float4*>(tabE + i * 4);
        e[0] = v.x; e[1] = v.y; e[2] = v.z; e[3] = v.w;
    }
}

// The per-cell range partials of a call that the contraction takes (the passes that record the
// table mode read them).
__device__ inline void sep_write_partials(const SepHead& h, const PrepArgs& p) {
    for (int i = threadIdx.x; i < kPrepBlocksX + kPrepBlocksW; i += blockDim.x) {
        float2 v = make_float2(INFINITY, -INFINITY);
        if (i == 0) v = make_float2(fmaf(h.xlo - p.xoff, p.scale, p.xadd), fmaf(h.xhi - p.xoff, p.scale, p.xadd));
        if (i == kPrepBlocksX) v = make_float2(h.wlo * p.scale, h.whi * p.scale);
        p.partials[i] = v;
    }
    if (p.stat_bits && threadIdx.x == 0) *p.stat_bits = 0u;
}

// Where the per-cell kernels take the call: their prep, in the same launch (unless the statistics'
// launch has run it).
__global__ __launch_bounds__(256) void sep_expand_fwd_kernel(SepArgs a, PrepArgs prep) {
    if (!sep_takes(a.head)) {
        if (blockIdx.x < kPrepBlocksX + kPrepBlocksW && a.head->rough != 2) prep_block(prep, blockIdx.x);
        return;
    }
    const SepHead h = *a.head;
    const int R = h.terms;
    if (blockIdx.x == 0) sep_write_partials(h, prep);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t kc = sep_inputs(a.K), pairs = sep_slabs_pairs(a.K, R) * 64;
    const int64_t stride = pairs + sep_slabs_singles(a.K, R, h.harmonics) * 64;  // of a row, in f16
    const int64_t harm = pairs + kc * (R / 2);
    const int64_t row_waves = (int64_t)gridDim.x * 4;
    const float as = a.in_affine ? a.in_affine[0] : 1.0f, ab = a.in_affine ? a.in_affine[1] : 0.0f;
    float v[4];
    for (int64_t row = (int64_t)blockIdx.x * 4 + wave; row < a.M + a.O; row += row_waves) {
        if (row < a.M) {
            float inv;
            const float scale = sep_scale_of(sep_bound(h, a.tab, 0, a.xrow[row], (float)a.v_sat), &inv);
            if (lane == 0) a.xscale[row] = inv / kSepQScale;
            _Float16* dst = a.xop + row * stride;
            for (int64_t k = lane; k < kc; k += 64) {
                const bool real = k < a.K;
                const float x = sep_input(a, a.x[row * a.K + (real ? k : a.K - 1)], as, ab);
                const float sc = real ? scale : 0.0f;
                const SepAt at = sep_at(h, x);
                for (int j = 0; j < R; j += 4) {
                    const float4 c = sep_eval4(a.tab, R, at, j);
                    v[0] = c.x * sc; v[1] = c.y * sc; v[2] = c.z * sc; v[3] = c.w * sc;
                    if (j < R / 2)
                        sep_store4(dst, j * kc + k * 4, v);
                    else
                        sep_store4h(dst + pairs, (j - R / 2) * kc + k * 4, v);
                }
                if (h.harmonics > 0) {
                    float e[4], c[2], sn[2];
                    sep_second(h, a.tabE, at, e);
                    sep_trig((x - h.lut_min) * h.lut_scale, c, sn);
                    for (int blk = 0; blk < h.harmonics * R / 8; ++blk) {
                        sep_harm_x(v, e, R, blk, c, sn, sc);
                        sep_store4h(dst + harm, blk * 4 * kc + k * 4, v);
                    }
                }
            }
        } else {
            const int64_t o = row - a.M;
            _Float16* dst = a.wop + o * stride;
            for (int64_t k = lane; k < kc; k += 64) {
                const bool real = k < a.K;
                const double tp = real ? ((double)a.wp[o * a.K + k] - h.wc) * h.inv_wh : 0.0;
                const double tn = real ? ((double)a.wn[o * a.K + k] - h.wc) * h.inv_wh : 0.0;
                SepChebPair c(tp, tn);
                for (int j = 0; j < R; j += 4) {
                    c.next4(v, kSepQScale);
                    if (j < R / 2)
                        sep_store4(dst, j * kc + k * 4, v);
                    else
                        sep_store4h(dst + pairs, (j - R / 2) * kc + k * 4, v);
                }
                if (h.harmonics > 0) {
                    float p[4], n[4], cp[2], sp[2], cn[2], sn[2];
                    sep_cheb4((float)tp, p);
                    sep_cheb4((float)tn, n);
                    sep_trig((float)((h.wc + h.wh * tp) * h.lut_scale), cp, sp);
                    sep_trig((float)((h.wc + h.wh * tn) * h.lut_scale), cn, sn);
                    for (int blk = 0; blk < h.harmonics * R / 8; ++blk) {
                        sep_harm_w(v, p, n, R, blk, cp, sp, cn, sn, kSepQScale);
                        sep_store4h(dst + harm, blk * 4 * kc + k * 4, v);
                    }
                }
            }
        }
    }
}

// ----------------------------------------------------------------------------------
// Backward operands, tokens or outputs inside: xop[(k, j)][m] = d_j r, wop[(k, j)][o] = T_j(t+) -
// T_j(t-) with tT[k][o] = {t+, t-}, gop[m][o] and gopT[o][m]. Tiles of 32 inputs (or rows of G)
// by 128 inner elements go through LDS, so that reads run along the tensors' rows and writes
// along the inner index. HBM-bound.
// ----------------------------------------------------------------------------------

__device__ inline void sep_store2h(_Float16* row, int64_t e, float v0, float v1) {  // single f16
    sep_h2 h;
    h.x = (_Float16)v0;
    h.y = (_Float16)v1;
    *reinterpret_cast<sep_h2*>(row + e) = h;
}

__global__ __launch_bounds__(256) void sep_expand_bwd_kernel(SepArgs a, int x_blocks, int w_blocks, PrepArgs prep) {
    if (!sep_takes(a.head)) {  // the per-cell kernels take the call: their prep
        if (blockIdx.x < kPrepBlocksX + kPrepBlocksW && a.head->rough != 2) prep_block(prep, blockIdx.x);
        return;
    }
    const SepHead h = *a.head;
    const int R = h.terms;
    if (blockIdx.x == 0) sep_write_partials(h, prep);
    const int64_t m64 = sep_slabs64(a.M) * 64, o64 = sep_slabs64(a.O) * 64;  // the singles' inner lengths
    const int xpairs = a.lut_n > 0 ? R / 2 : R;  // terms of xop as pairs
    __shared__ float s_a[32][130], s_b[32][130];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int64_t m_slabs = sep_slabs(a.M), o_slabs = sep_slabs(a.O);
    int b = blockIdx.x;
    if (b < x_blocks) {
        const int n_mt = (int)((a.M + 127) / 128);
        const int64_t m0 = (int64_t)(b % n_mt) * 128, k0 = (int64_t)(b / n_mt) * 32;
        const float as = a.in_affine ? a.in_affine[0] : 1.0f, ab = a.in_affine ? a.in_affine[1] : 0.0f;
        for (int q = t; q < 32 * 128; q += 256) {
            const int64_t m = m0 + (q >> 5), k = k0 + (q & 31);
            s_a[q & 31][q >> 5] = m < a.M && k < a.K ? sep_input(a, a.x[m * a.K + k], as, ab) : 0.0f;
        }
        __syncthreads();
        for (int kk = wave; kk < 32 && k0 + kk < a.K; kk += 4) {
            const int64_t k = k0 + kk;
            static_assert(kSepColChunks == 64, "a lane per chunk");
            float2 range = a.xcol[(int64_t)lane * a.K + k];
            sep_wave_minmax(range.x, range.y);
            float inv;
            const float scale = sep_scale_of(2.0f * sep_bound(h, a.tab, 0, range, (float)a.v_sat), &inv);
            if (m0 == 0 && lane == 0) a.xscale[k] = inv;
            const int ml = 2 * lane;
            const int64_t m = m0 + ml;
            if (m >= m64) continue;
            const bool pair = m < m_slabs * 32;
            const float s0 = m < a.M ? scale : 0.0f, s1 = m + 1 < a.M ? scale : 0.0f;
            const float x0 = m < a.M ? s_a[kk][ml] : range.y, x1 = m + 1 < a.M ? s_a[kk][ml + 1] : range.y;
            const SepAt p0 = sep_at(h, x0), p1 = sep_at(h, x1);
            for (int j = 0; j < R; j += 4) {
                const float4 u = sep_eval4(a.tab, R, p0, j), v = sep_eval4(a.tab, R, p1, j);
                const float u4[4] = {u.x * s0, u.y * s0, u.z * s0, u.w * s0}, v4[4] = {v.x * s1, v.y * s1, v.z * s1, v.w * s1};
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if (j < xpairs) {
                        if (pair) sep_store2(a.xop + sep_row(k, xpairs, j + q) * m_slabs * 64, m, u4[q], v4[q]);
                    } else {
                        sep_store2h(a.xops + sep_row(k, R / 2, j + q - R / 2) * m64, m, u4[q], v4[q]);
                    }
                }
            }
            if (h.harmonics > 0) {
                float e0[4], e1[4], c0[2], n0[2], c1[2], n1[2], u[4], v[4];
                sep_second(h, a.tabE, p0, e0);
                sep_second(h, a.tabE, p1, e1);
                sep_trig((x0 - h.lut_min) * h.lut_scale, c0, n0);
                sep_trig((x1 - h.lut_min) * h.lut_scale, c1, n1);
                for (int blk = 0; blk < h.harmonics * R / 8; ++blk) {
                    sep_harm_x(u, e0, R, blk, c0, n0, s0);
                    sep_harm_x(v, e1, R, blk, c1, n1, s1);
#pragma unroll
                    for (int q = 0; q < 4; ++q) sep_store2h(a.xoph + sep_row(k, h.harmonics * R / 2, blk * 4 + q) * m64, m, u[q], v[q]);
                }
            }
        }
        return;
    }
    b -= x_blocks;
    if (b < w_blocks) {
        const int n_ot = (int)((a.O + 127) / 128);
        const int64_t o0 = (int64_t)(b % n_ot) * 128, k0 = (int64_t)(b / n_ot) * 32;
        for (int q = t; q < 32 * 128; q += 256) {
            const int64_t o = o0 + (q >> 5), k = k0 + (q & 31);
            const bool real = o < a.O && k < a.K;
            s_a[q & 31][q >> 5] = real ? a.wp[o * a.K + k] : (float)h.wc;
            s_b[q & 31][q >> 5] = real ? a.wn[o * a.K + k] : (float)h.wc;
        }
        __syncthreads();
        for (int kk = wave; kk < 32 && k0 + kk < a.K; kk += 4) {
            const int64_t k = k0 + kk;
            const int ol = 2 * lane;
            const int64_t o = o0 + ol;
            if (o >= o64) continue;
            const bool pair = o < o_slabs * 32;
            double t_[4];
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                t_[2 * q] = ((double)s_a[kk][ol + q] - h.wc) * h.inv_wh;
                t_[2 * q + 1] = ((double)s_b[kk][ol + q] - h.wc) * h.inv_wh;
            }
            if (a.need_w) {
                reinterpret_cast<float4*>(a.tT + k * a.Op)[o >> 1] =
                    make_float4((float)t_[0], (float)t_[1], (float)t_[2], (float)t_[3]);
            }
            if (!a.need_x) continue;
            // padded outputs: both branches at the centre, so that their differences vanish
            SepChebPair c0(t_[0], t_[1]), c1(t_[2], t_[3]);
            float u[4], v[4];
            for (int j = 0; j < R; j += 4) {
                c0.next4(u, kSepQScale);
                c1.next4(v, kSepQScale);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if (j < R / 2) {
                        if (pair) sep_store2(a.wop + sep_row(k, R / 2, j + q) * o_slabs * 64, o, u[q], v[q]);
                    } else {
                        sep_store2h(a.wops + sep_row(k, R / 2, j + q - R / 2) * o64, o, u[q], v[q]);
                    }
                }
            }
            if (h.harmonics_dx > 0) {
                float p0[4], n0[4], p1[4], n1[4], e0[4], d0[4], e1[4], d1[4];
                sep_cheb4((float)t_[0], p0);
                sep_cheb4((float)t_[1], n0);
                sep_cheb4((float)t_[2], p1);
                sep_cheb4((float)t_[3], n1);
                sep_trig(s_a[kk][ol] * h.lut_scale, e0, d0);
                sep_trig(s_b[kk][ol] * h.lut_scale, e0 + 2, d0 + 2);
                sep_trig(s_a[kk][ol + 1] * h.lut_scale, e1, d1);
                sep_trig(s_b[kk][ol + 1] * h.lut_scale, e1 + 2, d1 + 2);
                for (int blk = 0; blk < h.harmonics_dx * R / 8; ++blk) {
                    sep_harm_w(u, p0, n0, R, blk, e0, d0, e0 + 2, d0 + 2, kSepQScale);
                    sep_harm_w(v, p1, n1, R, blk, e1, d1, e1 + 2, d1 + 2, kSepQScale);
#pragma unroll
                    for (int q = 0; q < 4; ++q) sep_store2h(a.woph + sep_row(k, h.harmonics_dx * R / 2, blk * 4 + q) * o64, o, u[q], v[q]);
                }
            }
        }
        return;
    }
    b -= w_blocks;
    if (b >= (int)((a.O + 127) / 128 * ((a.M + 31) / 32))) return;  // blocks that only the prep needs
    // G: tiles of 32 rows by 128 outputs
    const int n_ot = (int)((a.O + 127) / 128);
    const int64_t o0 = (int64_t)(b % n_ot) * 128, m0 = (int64_t)(b / n_ot) * 32;
    for (int q = t; q < 32 * 128; q += 256) {
        const int64_t m = m0 + (q >> 7), o = o0 + (q & 127);
        s_a[q >> 7][q & 127] = m < a.M && o < a.O ? a.g[m * a.ldg + o] : 0.0f;
    }
    __syncthreads();
    if (a.need_x) {
        for (int mm = wave; mm < 32 && m0 + mm < a.M; mm += 4) {
            const int64_t m = m0 + mm, o = o0 + 2 * lane;
            float inv;
            const float scale = sep_scale_of(__uint_as_float(a.grow[m]), &inv);
            if (o0 == 0 && lane == 0) a.gscale[m] = inv / kSepQScale;
            const float g0 = s_a[mm][2 * lane] * scale, g1 = s_a[mm][2 * lane + 1] * scale;
            if (o < o_slabs * 32) sep_store2(a.gop + m * o_slabs * 64, o, g0, g1);
            if (o < o64) sep_store2h(a.goph + m * o64, o, g0, g1);
        }
    }
    if (a.need_w) {
        // 16 lanes hold the 32 tokens of one output: 16 outputs at a time
        for (int q = t >> 4; q < 128 && o0 + q < a.O; q += 16) {
            const int64_t o = o0 + q;
            unsigned big = 0;
            for (int c = t & 15; c < kSepColChunks; c += 16) big = max(big, a.gcol[(int64_t)c * a.O + o]);
            for (int d = 8; d > 0; d >>= 1) big = max(big, (unsigned)__shfl_xor((int)big, d, 16));
            float inv;
            const float scale = sep_scale_of(__uint_as_float(big), &inv);
            if (m0 == 0 && (t & 15) == 0) a.gscaleT[o] = inv;
            const int mm = 2 * (t & 15);
            const float g0 = s_a[mm][q] * scale, g1 = s_a[mm + 1][q] * scale;
            sep_store2(a.gopT + o * m_slabs * 64, m0 + mm, g0, g1);
            sep_store2h(a.gophT + o * m64, m0 + mm, g0, g1);
            if (m0 + 32 >= a.M && m0 + 32 < m64) sep_store2h(a.gophT + o * m64, m0 + 32 + mm, 0.0f, 0.0f);
        }
    }
}

// ----------------------------------------------------------------------------------
// The product of two operands of slabs, C[i][j] = sum_e A[i][e] B[j][e]: tiles of
// (WM MI 32) x (WN NI 32), one slab (128 bytes per row) of both operands at a time in two LDS
// buffers. A slab holds 32 inner elements as hi/lo pairs, which take three products per pair of
// fragments (hi hi, hi lo, lo hi), or (harmonics) 64 as single f16. A slab's loads are issued
// before the arithmetic of the one before it: 3072 matrix-core cycles per 64 KB of operands for
// the 256 x 256 tile of pairs, so that one buffer ahead covers the memory's latency and the
// operands need ~21 bytes per cycle and CU. Rows are 128 bytes and their eight 16-byte parts are
// stored at part ^ (row / 2 % 8), so that the 16 rows that a quarter-wave reads lie on different
// banks. Rows past the operand's end read its last row (their results are dropped).
// Blocks are dealt so that each XCD works on neighbouring tiles (whose operands its L2 holds).
//
// A launch runs up to six products after one another in its grid (the backward's dX and dVth, of
// the lower terms, the upper ones and the harmonics), so that one's last blocks overlap the next one's first.
// ----------------------------------------------------------------------------------

enum SepKind { kSepForward, kSepDx, kSepDv, kSepDxUpper, kSepDvUpper, kSepDxHarm, kSepDvHarm };

struct SepProduct {
    const char* a;
    const char* b;
    int kind;
    int64_t a_rows, b_rows;   // dX, dVth: inputs in the place of A's rows
    int64_t inner;            // elements; forward: inputs
    int n_split;
    float* out;               // forward: planes [n_split][M][O]; dX: [n_split][M][K]; dVth: [n_split][2][Kp][Op]
};

struct SepGemm {
    SepProduct p[6];
    int n;
    const SepHead* head;
    int64_t M, K, O, Kp, Op;
    const float* xscale;      // forward [M], dVth [K]
    const float* gscale;      // dX [M]
    const float* gscaleT;     // dVth [O]
    const float* x;
    const float* in_affine;
    float in_lo, in_hi;
    const float* tab2;
    const float* tabE;
    const float2* tT;
    int dv_all;               // the dVth product of pairs holds every term
};

template <int WM, int WN, int MI, int NI, bool FORWARD>
__global__ __launch_bounds__(WM * WN * 64, 2) void sep_gemm_kernel(SepGemm g) {
    constexpr int kThreads = WM * WN * 64, TM = WM * MI * 32, TN = WN * NI * 32;
    constexpr int kLoadA = TM * 8 / kThreads, kLoadB = TN * 8 / kThreads, kRowStep = kThreads / 8;
    extern __shared__ __attribute__((aligned(16))) char s_sep[];
    const SepHead* head = g.head;
    if (!sep_takes(head)) return;
    const int R = __builtin_amdgcn_readfirstlane(head->terms);
    const int harmonics = __builtin_amdgcn_readfirstlane(head->harmonics);
    const int harmonics_dx = FORWARD ? 0 : __builtin_amdgcn_readfirstlane(head->harmonics_dx);
    // the product this block works on, its rows and slabs, and the blocks of four values per input
    int id = blockIdx.x, which = 0, ta = 0, tb = 0, n = 0, slabs = 0, pair_slabs = 0, per = 0;
    int64_t a_rows = 0;
    for (;; ++which) {
        if (which >= g.n) return;
        const SepProduct& p = g.p[which];
        if constexpr (FORWARD) {
            a_rows = p.a_rows;
            pair_slabs = (int)sep_slabs_pairs(p.inner, R);
            slabs = pair_slabs + (int)sep_slabs_singles(p.inner, R, harmonics);
        } else {
            const bool pairs = p.kind == kSepDx || p.kind == kSepDv;
            per = p.kind == kSepDxHarm             ? harmonics_dx * R / 8
                  : p.kind == kSepDvHarm           ? harmonics * R / 8
                  : p.kind == kSepDv && g.dv_all ? R / 4
                                                   : R / 8;
            a_rows = (p.a_rows + 1) / 2 * 8 * per;
            slabs = (int)(pairs ? sep_slabs(p.inner) : sep_slabs64(p.inner));
            pair_slabs = pairs ? slabs : 0;
        }
        ta = (int)((a_rows + TM - 1) / TM);
        tb = (int)((p.b_rows + TN - 1) / TN);
        n = ta * tb * p.n_split;
        if (id < n) break;
        id -= n;
    }
    const SepProduct& p = g.p[which];
    {   // blocks run over the XCDs round robin: give XCD c the tiles [c n / 8, (c + 1) n / 8)
        const int per = n / 8, rest = n % 8, xcd = id & 7;
        id = xcd * per + (xcd < rest ? xcd : rest) + (id >> 3);
    }
    // tiles of one split in groups of four along A: neighbours share both operands
    const int split = id / (ta * tb);
    id -= split * (ta * tb);
    const int group = id / (4 * tb), in_group = id - group * 4 * tb;
    const int height = min(4, ta - group * 4);
    const int tile_a = group * 4 + in_group % height, tile_b = in_group / height;
    const int64_t a0 = (int64_t)tile_a * TM, b0 = (int64_t)tile_b * TN;
    const int s_begin = (int)((int64_t)slabs * split / p.n_split);
    const int s_end = (int)((int64_t)slabs * (split + 1) / p.n_split);

    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int wr = wave / WN, wc = wave % WN;
    const int row0 = t >> 3, part = (t & 7) ^ ((row0 >> 1) & 7);
    unsigned pa[kLoadA], pb[kLoadB];  // byte offsets (an operand holds less than 4 GiB)
#pragma unroll
    for (int q = 0; q < kLoadA; ++q) {
        const int64_t row = a0 + row0 + q * kRowStep;
        pa[q] = (unsigned)(((row < a_rows ? row : a_rows - 1) * slabs * 8 + part) * 16);
    }
#pragma unroll
    for (int q = 0; q < kLoadB; ++q) {
        const int64_t row = b0 + row0 + q * kRowStep;
        pb[q] = (unsigned)(((row < p.b_rows ? row : p.b_rows - 1) * slabs * 8 + part) * 16);
    }
    constexpr int kBuf = (TM + TN) * 128;
    // kRowStep rows further on the swizzle is the same: kRowStep is a multiple of 16
    static_assert(kRowStep % 16 == 0, "");
    const int fl = lane & 31, fh = lane >> 5;
    const int frag = fl * 128 + ((fh ^ ((fl >> 1) & 7)) << 4);
    const int fa = wr * MI * 32 * 128, fb = TM * 128 + wc * NI * 32 * 128;

    sep_f16 acc[MI][NI];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j)
#pragma unroll
            for (int q = 0; q < 16; ++q) acc[i][j][q] = 0.0f;

    const char* abase = p.a;
    const char* bbase = p.b;
    // a wave's loads of a slab: eight rows of 128 bytes each, straight into LDS (lane i to byte
    // 16 i of the kilobyte): the lane that fills part p of a row reads part p ^ (row / 2 % 8)
    auto copy = [&](int s, int buf) {
        char* dst = s_sep + buf * kBuf + wave * 1024;
#pragma unroll
        for (int q = 0; q < kLoadA; ++q)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(abase + (pa[q] + (unsigned)s * 128u)),
                                             (__attribute__((address_space(3))) void*)(dst + q * kThreads * 16), 16, 0, 0);
#pragma unroll
        for (int q = 0; q < kLoadB; ++q)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(bbase + (pb[q] + (unsigned)s * 128u)),
                                             (__attribute__((address_space(3))) void*)(dst + TM * 128 + q * kThreads * 16), 16, 0, 0);
    };
    auto multiply = [&](const sep_h8* u, const sep_h8* v) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NI; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(u[i], v[j], acc[i][j], 0, 0, 0);
    };
    if (s_begin < s_end) copy(s_begin, 0);
    int s = s_begin;
    const int pair_end = min(s_end, pair_slabs);
    for (; s < pair_end; ++s) {
        const int buf = (s - s_begin) & 1;
        __syncthreads();  // this slab has landed, and the other buffer's has been read
        const char* base = s_sep + buf * kBuf;
        sep_h8 ah[2][MI], al[2][MI], bh[2][NI], bl[2][NI];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const int off = frag ^ (ks << 5);  // parts ks * 2 + fh (hi), + 4 (lo)
#pragma unroll
            for (int j = 0; j < NI; ++j) bh[ks][j] = *reinterpret_cast<const sep_h8*>(base + fb + j * 4096 + off);
#pragma unroll
            for (int i = 0; i < MI; ++i) ah[ks][i] = *reinterpret_cast<const sep_h8*>(base + fa + i * 4096 + off);
#pragma unroll
            for (int j = 0; j < NI; ++j) bl[ks][j] = *reinterpret_cast<const sep_h8*>(base + fb + j * 4096 + (off ^ 64));
#pragma unroll
            for (int i = 0; i < MI; ++i) al[ks][i] = *reinterpret_cast<const sep_h8*>(base + fa + i * 4096 + (off ^ 64));
        }
        if (s + 1 < s_end) copy(s + 1, buf ^ 1);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            multiply(ah[ks], bh[ks]);
            multiply(ah[ks], bl[ks]);
            multiply(al[ks], bh[ks]);
        }
    }
    for (; s < s_end; ++s) {
        const int buf = (s - s_begin) & 1;
        __syncthreads();
        const char* base = s_sep + buf * kBuf;
        sep_h8 av[4][MI], bv[4][NI];
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            const int off = frag ^ (ks << 5);
#pragma unroll
            for (int i = 0; i < MI; ++i) av[ks][i] = *reinterpret_cast<const sep_h8*>(base + fa + i * 4096 + off);
#pragma unroll
            for (int j = 0; j < NI; ++j) bv[ks][j] = *reinterpret_cast<const sep_h8*>(base + fb + j * 4096 + off);
        }
        if (s + 1 < s_end) copy(s + 1, buf ^ 1);
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) multiply(av[ks], bv[ks]);
    }

    // lane (fl, fh) holds rows q % 4 + 8 (q / 4) + 4 fh of column fl of each 32 x 32 tile
    if constexpr (FORWARD) {
        float* out = p.out + (int64_t)split * g.M * g.O;
#pragma unroll
        for (int i = 0; i < MI; ++i) {
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const int64_t m = a0 + (wr * MI + i) * 32 + (q & 3) + 8 * (q >> 2) + 4 * fh;
                if (m >= g.M) continue;
                const float sc = g.xscale[m];
#pragma unroll
                for (int j = 0; j < NI; ++j) {
                    const int64_t o = b0 + (wc * NI + j) * 32 + fl;
                    if (o < g.O) out[m * g.O + o] = acc[i][j][q] * sc;
                }
            }
        }
    } else {
        const SepHead h = *head;
        const int kind = p.kind;
        const bool harm = kind >= kSepDxHarm, upper = kind == kSepDxUpper || kind == kSepDvUpper;
        const int sh = __builtin_ctz(per), j_first = upper ? R / 2 : 0;
        const bool eight = R == 8;
        if (kind == kSepDx || kind == kSepDxUpper || kind == kSepDxHarm) {
            const float as = g.in_affine ? g.in_affine[0] : 1.0f, ab = g.in_affine ? g.in_affine[1] : 0.0f;
            float* out = p.out + (int64_t)split * g.M * g.K;
#pragma unroll
            for (int j = 0; j < NI; ++j) {
                const int64_t m = b0 + (wc * NI + j) * 32 + fl;
                const int64_t mc = m < g.M ? m : g.M - 1;
                const float sc = g.gscale[mc];
                float sum = 0.0f;
#pragma unroll
                for (int i = 0; i < MI; ++i) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) {  // block jb of inputs k (fh = 0) and k + 1
                        const int64_t block = (a0 + (wr * MI + i) * 32) / 8 + q;
                        const int64_t k = (block >> sh) * 2 + fh;
                        const int jb = (int)block & (per - 1);
                        const float xr = g.x[mc * g.K + (k < g.K ? k : g.K - 1)];
                        const float x = g.in_affine ? input_map(xr, as, ab, g.in_lo, g.in_hi) : xr;
                        const SepAt at = sep_at(h, x);
                        float4 v;
                        if (!harm) {
                            v = sep_eval4(g.tab2, R, at, j_first + 4 * jb);
                        } else {
                            const bool second = eight ? jb & 1 : jb & 2;
                            const float th = (x - h.lut_min) * h.lut_scale * (second ? 2.0f : 1.0f);
                            const float f = th - floorf(th), w = second ? 0.25f : 1.0f;
                            const float c = __builtin_amdgcn_cosf(f) * w, sn = __builtin_amdgcn_sinf(f) * w;
                            float e[4];
                            sep_second(h, g.tabE, at, e);
                            if (eight) {
                                v = make_float4(e[0] * c, e[1] * c, e[0] * sn, e[1] * sn);
                            } else {
                                const float tr = jb & 1 ? sn : c;
                                v = make_float4(e[0] * tr, e[1] * tr, e[2] * tr, e[3] * tr);
                            }
                        }
                        sum = fmaf(acc[i][j][4 * q], v.x, sum);
                        sum = fmaf(acc[i][j][4 * q + 1], v.y, sum);
                        sum = fmaf(acc[i][j][4 * q + 2], v.z, sum);
                        sum = fmaf(acc[i][j][4 * q + 3], v.w, sum);
                        if (jb == per - 1) {
                            if (m < g.M && k < g.K) out[m * g.K + k] = sum * sc;
                            sum = 0.0f;
                        }
                    }
                }
            }
        } else {
            float* out = p.out + (int64_t)split * 2 * g.Kp * g.Op;
#pragma unroll
            for (int j = 0; j < NI; ++j) {
                const int64_t o = b0 + (wc * NI + j) * 32 + fl;
                const int64_t oc = o < g.O ? o : g.O - 1;
                const float sb = g.gscaleT[oc];
                float sp = 0.0f, sn = 0.0f, p0 = 0.0f, p1 = 0.0f, n0 = 0.0f, n1 = 0.0f;
                float2 tt = make_float2(0.0f, 0.0f);
#pragma unroll
                for (int i = 0; i < MI; ++i) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const int64_t block = (a0 + (wr * MI + i) * 32) / 8 + q;
                        const int64_t k = (block >> sh) * 2 + fh;
                        const int jb = (int)block & (per - 1);
                        if (jb == 0) tt = g.tT[(k < g.K ? k : g.K - 1) * g.Op + oc];
                        const float a0_ = acc[i][j][4 * q], a1_ = acc[i][j][4 * q + 1], a2_ = acc[i][j][4 * q + 2],
                                    a3_ = acc[i][j][4 * q + 3];
                        float rp = 0.0f, rn = 0.0f;
                        if (!harm) {
                            if (jb == 0) {
                                if (!upper) {  // T_0, T_1
                                    p0 = n0 = 1.0f;
                                    p1 = tt.x;
                                    n1 = tt.y;
                                } else {  // T_(R/2), T_(R/2 + 1) = cos(j acos t): 1e-5, of terms below 4e-3
                                    const float u = acosf(fminf(fmaxf(tt.x, -1.0f), 1.0f)) * 0.15915494f;
                                    const float w = acosf(fminf(fmaxf(tt.y, -1.0f), 1.0f)) * 0.15915494f;
                                    const float jf = (float)j_first;
                                    auto cosj = [](float r) { return __builtin_amdgcn_cosf(r - floorf(r)); };
                                    p0 = cosj(u * jf);
                                    p1 = cosj(u * (jf + 1.0f));
                                    n0 = cosj(w * jf);
                                    n1 = cosj(w * (jf + 1.0f));
                                }
                            }
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                rp = fmaf(acc[i][j][4 * q + e], p0, rp);
                                rn = fmaf(acc[i][j][4 * q + e], n0, rn);
                                const float p2 = fmaf(2.0f * tt.x, p1, -p0), n2 = fmaf(2.0f * tt.y, n1, -n0);
                                p0 = p1;
                                p1 = p2;
                                n0 = n1;
                                n1 = n2;
                            }
                        } else {
                            const bool second = eight ? jb & 1 : jb & 2;
                            const float ws = h.lut_scale * (second ? 2.0f : 1.0f);
                            const float tp = ((float)h.wc + (float)h.wh * tt.x) * ws, tn = ((float)h.wc + (float)h.wh * tt.y) * ws;
                            const float fp = tp - floorf(tp), fn = tn - floorf(tn);
                            const float cp = __builtin_amdgcn_cosf(fp), dp = __builtin_amdgcn_sinf(fp);
                            const float cn = __builtin_amdgcn_cosf(fn), dn = __builtin_amdgcn_sinf(fn);
                            if (eight) {
                                rp = cp * fmaf(a1_, tt.x, a0_) + dp * fmaf(a3_, tt.x, a2_);
                                rn = cn * fmaf(a1_, tt.y, a0_) + dn * fmaf(a3_, tt.y, a2_);
                            } else {
                                float vp[4], vn[4];
                                sep_cheb4(tt.x, vp);
                                sep_cheb4(tt.y, vn);
                                rp = (jb & 1 ? dp : cp) * fmaf(a3_, vp[3], fmaf(a2_, vp[2], fmaf(a1_, vp[1], a0_)));
                                rn = (jb & 1 ? dn : cn) * fmaf(a3_, vn[3], fmaf(a2_, vn[2], fmaf(a1_, vn[1], a0_)));
                            }
                        }
                        sp += rp;
                        sn += rn;
                        if (jb == per - 1) {
                            if (o < g.O && k < g.K) {
                                const float sc = sb * g.xscale[k];
                                out[k * g.Op + o] = sp * sc;
                                out[(g.Kp + k) * g.Op + o] = sn * sc;
                            }
                            sp = sn = 0.0f;
                        }
                    }
                }
            }
        }
    }
}

// Finishes the forward (split_reduce_body) from the planes of whichever path took the call; a
// per-cell plan without a split (cell.n_split <= 1) has written its outputs itself.
template <int VEC>
__global__ __launch_bounds__(256) void sep_reduce_fwd_kernel(FwdArgs sep, FwdArgs cell, const SepHead* head,
                                                             int clamp_out) {
    if (sep_takes(head))
        split_reduce_body<VEC>(sep, clamp_out);
    else if (cell.n_split > 1)
        split_reduce_body<VEC>(cell, clamp_out);
}

// grad_reduce_kernel's work from the planes of whichever path took the call.
__global__ __launch_bounds__(256) void sep_reduce_bwd_kernel(DxReduceArgs dx, DxReduceArgs dx_cell, int dx_blocks,
                                                             DvReduceArgs dv, DvReduceArgs dv_cell, int dv_blocks,
                                                             GlueReduceArgs gl, const SepHead* head, int harm_dx,
                                                             int harm_dv) {
    const int b = blockIdx.x;
    if (b >= dx_blocks + dv_blocks) {
        glue_reduce_block(gl, b - dx_blocks - dv_blocks);
        return;
    }
    if (sep_takes(head)) {
        if (head->harmonics == 0) {  // their planes, the last ones, were not written
            dx.n_planes -= harm_dx;
            dv.n_split -= harm_dv;
        }
        if (b < dx_blocks)
            dx_reduce_block(dx, b, dx_blocks);
        else
            dv_reduce_block(dv, b - dx_blocks, dv_blocks);
    } else {
        if (b < dx_blocks)
            dx_reduce_block(dx_cell, b, dx_blocks);
        else
            dv_reduce_block(dv_cell, b - dx_blocks, dv_blocks);
    }
}

// ----------------------------------------------------------------------------------
// Host side: plans and launches.
// ----------------------------------------------------------------------------------

// Calls of fewer cells M K O run the per-cell kernels. A call that the contraction refuses pays for
// the launches that return, 14 us where the sample refuses it (sep_sample_refuses; 5 us less for
// tables, whose assignment passes are one launch), and the statistics, 11 us, where only they do:
// the lines lie where that is 1% of the call. Measured (us, forward and backward, without the
// contraction against refused): formula, 192 x 768 over 2 V at 2^27.2 cells 444 against 458, at
// 2^28 over 4 V 804 against 820; tables over 5 V at 2^29 614 against 626, 768 -> 3072 -> 768 at
// 2048 tokens (two calls of 2^32.2) 9125 against 9135. Taken calls gain from far smaller sizes on:
// formula, 192 x 768 at 2^25.2 164 against 153, at 2^27.2 444 against 156.
#ifndef ISA_EKV_CONTRACT_MIN_CELLS
#define ISA_EKV_CONTRACT_MIN_CELLS (1 << 29)
#endif
// Table calls (us, forward / backward, per-cell kernels against the contraction, 4096 entries):
// 384 x 1536 at 2^30 cells 334 / 557 against 137 / 261 at the initial thresholds, 344 / 740 against
// 222 / 398 over 1 V (16 terms), 399 / 783 against 410 / 791 over 5 V (refused); at 2^29 224 / 329
// against 98 / 200, 219 / 414 against 142 / 296, and 237 / 462 against 246 / 472.
#ifndef ISA_EKV_CONTRACT_MIN_CELLS_LUT
#define ISA_EKV_CONTRACT_MIN_CELLS_LUT (1 << 30)
#endif

struct SepPlan {
    int max_terms;  // 0: not considered
    bool big;       // 256 x 256 tiles instead of 128 x 128
    int split, split_dx, split_dv, split_dxs, split_dvs, split_dxh, split_dvh;
    int planes_dx, planes_dv;
    int64_t Kp, Op;
    size_t off_head, off_part, off_row, off_col, off_grow, off_gcol, off_tab, off_tab2, off_tabE, off_lut, off_xop, off_wop,
        off_xops, off_wops, off_xoph, off_woph, off_gop, off_gopT, off_goph, off_gophT, off_scale, off_gscale, off_gscaleT, off_tT,
        off_planes, off_planes_dv, bytes;
};

constexpr int64_t kSepOperandBytes = (int64_t)2 << 30;  // of one operand, at most (32-bit byte offsets)

// Splits of a product's inner length: the count (each at least 8 slabs) that makes the launch's
// time least, in slabs of one tile: rounds of blocks over the CUs (one 256 x 256 block each,
// two of 128 x 128), each the split's slabs and about 5 more of prologue and epilogue, and for
// every further plane its write and read back against ~1.4 us a slab.
inline int sep_splits(int64_t tiles, int64_t slabs, bool big, double plane_bytes) {
    int best = 1;
    double best_cost = 0.0;
    const int64_t at_once = big ? kCUs : 2 * kCUs;
    for (int s = 1; s <= 16 && (s == 1 || slabs / s >= 8); ++s) {
        const double rounds = (double)((tiles * s + at_once - 1) / at_once);
        const double cost = rounds * ((double)(slabs + s - 1) / s + 5.0) + s * plane_bytes / 4e12 / (big ? 1.4e-6 : 0.7e-6);
        if (s == 1 || cost < best_cost) {
            best = s;
            best_cost = cost;
        }
    }
    return best;
}

inline bool sep_big(int64_t rows_a, int64_t rows_b, int64_t slabs) {
    // 256 x 256 tiles halve the operand reads per product; they need enough of them
    return ((rows_a + 255) / 256) * ((rows_b + 255) / 256) * (slabs / 16 + 1) >= 2 * kCUs && rows_a >= 192 && rows_b >= 192;
}

// lut_n: table entries, 0 for the formula.
SepPlan plan_sep(int lut_n, int64_t M, int64_t K, int64_t O, bool backward, bool need_x, bool need_w, size_t base) {
    SepPlan p{};
    p.bytes = base;
    const double cells = (double)M * (double)K * (double)O;
    if (M < 16 || O < 16 || K < 8 || (backward && !need_x && !need_w) ||
        cells < (double)(lut_n > 0 ? (int64_t)ISA_EKV_CONTRACT_MIN_CELLS_LUT : (int64_t)ISA_EKV_CONTRACT_MIN_CELLS) ||
        (lut_n > 0 && (lut_n < kSepLutMin || lut_n > kSepLutMax)))
        return p;
    p.Kp = round_up(K, 8);
    p.Op = round_up(O, 256);
    const int64_t Mr = round_up(M, 64), Or = round_up(O, 64), Kr = sep_inputs(K);
    const int harm = lut_n > 0 ? 1 : 0;
    // bytes per (row, input), forward: R / 2 pairs, R / 2 singles and the harmonics; an operand's
    // size backward: at most R pairs
    auto width = [&](int terms) { return (int64_t)terms * (backward ? 4 : 3 + 2 * harm); };
    int terms = kSepMaxTerms;
    while (terms >= 8 && (Mr * Kr * width(terms) >= kSepOperandBytes || Or * Kr * width(terms) >= kSepOperandBytes)) terms /= 2;
    if (terms < 8 || Mr * Or * 4 >= kSepOperandBytes) return p;
    p.max_terms = terms;
    size_t off = (size_t)round_up((int64_t)base, 256);
    auto take = [&](int64_t bytes) {
        const size_t at = off;
        off += (size_t)round_up(bytes, 256);
        return at;
    };
    p.off_head = take(sizeof(SepHead));
    p.off_part = take((kSepStatX + kSepStatW) * 8);
    p.off_tab = take((int64_t)kSepGridMax * 4 * terms);
    if (lut_n > 0) {
        p.off_lut = take((int64_t)lut_n * 16 + 256 * 8);
        p.off_tabE = take((int64_t)kSepGridMax * terms);
    }
    if (!backward) {
        p.off_xop = take(Mr * Kr * width(terms));
        p.off_wop = take(Or * Kr * width(terms));
        p.off_row = take(M * 8);
        p.off_scale = take(M * 4);
        const int64_t slabs = sep_slabs_pairs(K, 8) + sep_slabs_singles(K, 8, harm);
        p.big = sep_big(M, O, slabs);
        const int64_t tile = p.big ? 256 : 128;
        p.split = sep_splits(((M + tile - 1) / tile) * ((O + tile - 1) / tile), slabs, p.big, 8.0 * M * O);
        p.off_planes = take((int64_t)p.split * M * O * 4);
    } else {
        p.off_tab2 = take((int64_t)kSepGridMax * 4 * terms);
        p.off_col = take(kSepColChunks * K * 8);
        p.off_grow = take(M * 4);
        p.off_gcol = take(kSepColChunks * O * 4);
        p.off_gop = take(Mr * Or * 4);
        p.off_gopT = take(Mr * Or * 4);
        p.off_goph = take(Mr * Or * 2);
        p.off_gophT = take(Mr * Or * 2);
        if (need_w) p.off_xop = take(Mr * Kr * terms * (harm ? 2 : 4));
        if (need_w && harm) p.off_xops = take(Mr * Kr * terms);
        if (need_w && harm) p.off_xoph = take(Mr * Kr * terms * 2);
        if (need_x) {
            p.off_wop = take(Or * Kr * terms * 2);
            p.off_wops = take(Or * Kr * terms);
            if (harm) p.off_woph = take(Or * Kr * terms * 2);
        }
        p.off_scale = take(K * 4);
        p.off_gscale = take(M * 4);
        p.off_gscaleT = take(O * 4);
        p.off_tT = take(K * p.Op * 8);
        p.big = sep_big(8 * K, std::min(M, O), std::min(M, O) / 32);
        // at 8 terms: 4 rows per input of lower and of upper terms (8 of the formula's dVth), 4 of a harmonic
        // (dX has two below ~6000 entries)
        const int64_t tile = p.big ? 256 : 128, t4 = (4 * K + tile - 1) / tile, t8 = (8 * K + tile - 1) / tile;
        const int64_t tm = (M + tile - 1) / tile, to = (O + tile - 1) / tile;
        const double dx_bytes = 8.0 * M * K, dv_bytes = 16.0 * p.Kp * p.Op;
        p.split_dx = sep_splits(t4 * tm, (O + 31) / 32, p.big, dx_bytes);
        p.split_dxs = sep_splits(t4 * tm, (O + 63) / 64, p.big, dx_bytes);
        p.split_dv = sep_splits((harm ? t4 : t8) * to, (M + 31) / 32, p.big, dv_bytes);
        p.split_dvs = harm ? sep_splits(t4 * to, (M + 63) / 64, p.big, dv_bytes) : 0;
        p.split_dxh = harm ? sep_splits((lut_n < 6000 ? t8 : t4) * tm, (O + 63) / 64, p.big, dx_bytes) : 0;
        p.split_dvh = harm ? sep_splits(t4 * to, (M + 63) / 64, p.big, dv_bytes) : 0;
        p.planes_dx = p.split_dx + p.split_dxs + p.split_dxh;
        p.planes_dv = p.split_dv + p.split_dvs + p.split_dvh;
        if (need_x) p.off_planes = take((int64_t)p.planes_dx * M * K * 4);
        if (need_w) p.off_planes_dv = take((int64_t)p.planes_dv * 2 * p.Kp * p.Op * 4);
    }
    p.bytes = off;
    return p;
}

template <bool FORWARD>
void launch_sep_gemm(bool big, unsigned blocks, const SepGemm& g, hipStream_t s) {
    if (big)
        hipLaunchKernelGGL((sep_gemm_kernel<2, 4, 4, 2, FORWARD>), dim3(blocks), dim3(512), 131072, s, g);
    else
        hipLaunchKernelGGL((sep_gemm_kernel<2, 2, 2, 2, FORWARD>), dim3(blocks), dim3(256), 65536, s, g);
}

void sep_point(const SepPlan& p, SepArgs& a, char* ws) {
    a.head = reinterpret_cast<SepHead*>(ws + p.off_head);
    a.xpart = reinterpret_cast<float2*>(ws + p.off_part);
    a.wpart = a.xpart + kSepStatX;
    a.tab = reinterpret_cast<float*>(ws + p.off_tab);
    a.tabE = reinterpret_cast<float*>(ws + p.off_tabE);
    a.lut_info = reinterpret_cast<float2*>(ws + p.off_lut);
    a.lut_val = reinterpret_cast<double2*>(ws + p.off_lut + 256 * 8);
    a.xop = reinterpret_cast<_Float16*>(ws + p.off_xop);
    a.wop = reinterpret_cast<_Float16*>(ws + p.off_wop);
    a.xscale = reinterpret_cast<float*>(ws + p.off_scale);
    a.max_terms = p.max_terms;
}

// The forward's operands (and, where it does not take the call, the per-cell kernels' prep).
hipError_t sep_forward_operands(const SepPlan& p, SepArgs a, const PrepArgs& prep, char* ws, hipStream_t s) {
    sep_point(p, a, ws);
    a.xrow = reinterpret_cast<float2*>(ws + p.off_row);
    hipLaunchKernelGGL(sep_stat_kernel, dim3(kSepStatX + kSepStatW + (a.lut_n + 255) / 256), dim3(256), 0, s, a,
                       prep, GlueGradArgs{});
    hipLaunchKernelGGL(sep_table_kernel, dim3(kSepTableBlocks), dim3(256), 0, s, a);
    const int64_t expand = std::min<int64_t>((a.M + a.O + 3) / 4, kSepExpandBlocks);
    hipLaunchKernelGGL(sep_expand_fwd_kernel, dim3((unsigned)std::max<int64_t>(expand, kPrepBlocksX + kPrepBlocksW)),
                       dim3(256), 0, s, a, prep);
    return hipGetLastError();
}

// The forward's product, into its planes.
hipError_t sep_forward_product(const SepPlan& p, SepArgs a, char* ws, hipStream_t s) {
    sep_point(p, a, ws);
    SepGemm g{};
    g.head = a.head;
    g.M = a.M;
    g.K = a.K;
    g.O = a.O;
    g.xscale = a.xscale;
    g.n = 1;
    g.p[0] = SepProduct{reinterpret_cast<const char*>(a.xop), reinterpret_cast<const char*>(a.wop), kSepForward, a.M, a.O,
                        a.K, p.split, reinterpret_cast<float*>(ws + p.off_planes)};
    const int64_t tile = p.big ? 256 : 128;
    launch_sep_gemm<true>(p.big, (unsigned)((a.M + tile - 1) / tile * ((a.O + tile - 1) / tile) * p.split), g, s);
    return hipGetLastError();
}

void sep_point_backward(const SepPlan& p, SepArgs& a, char* ws) {
    sep_point(p, a, ws);
    a.xcol = a.need_w ? reinterpret_cast<float2*>(ws + p.off_col) : nullptr;
    a.grow = reinterpret_cast<unsigned*>(ws + p.off_grow);
    a.gcol = reinterpret_cast<unsigned*>(ws + p.off_gcol);
    a.tab2 = reinterpret_cast<float*>(ws + p.off_tab2);
    a.gop = reinterpret_cast<_Float16*>(ws + p.off_gop);
    a.gopT = reinterpret_cast<_Float16*>(ws + p.off_gopT);
    a.xops = reinterpret_cast<_Float16*>(ws + p.off_xops);
    a.wops = reinterpret_cast<_Float16*>(ws + p.off_wops);
    a.xoph = reinterpret_cast<_Float16*>(ws + p.off_xoph);
    a.woph = reinterpret_cast<_Float16*>(ws + p.off_woph);
    a.goph = reinterpret_cast<_Float16*>(ws + p.off_goph);
    a.gophT = reinterpret_cast<_Float16*>(ws + p.off_gophT);
    a.gscale = reinterpret_cast<float*>(ws + p.off_gscale);
    a.gscaleT = reinterpret_cast<float*>(ws + p.off_gscaleT);
    a.tT = reinterpret_cast<float2*>(ws + p.off_tT);
    a.Op = p.Op;
}

// The backward's operands; glue: the layer glue's gradient pass, which writes a.g.
hipError_t sep_backward_operands(const SepPlan& p, SepArgs a, const PrepArgs& prep, const GlueGradArgs* glue, char* ws,
                                 hipStream_t s) {
    sep_point_backward(p, a, ws);
    const int64_t xcols = a.xcol ? kSepColChunks * ((a.K + 255) / 256) : 0;
    const int64_t stat = kSepStatX + kSepStatW + (a.lut_n + 255) / 256 + xcols + (glue ? (int64_t)kGlueBlocks * (glue->Op / 256) : 0);
    hipLaunchKernelGGL(sep_stat_kernel, dim3((unsigned)stat), dim3(256), 0, s, a, prep,
                       glue ? *glue : GlueGradArgs{});
    const int64_t gcols = a.need_w ? kSepColChunks * ((a.O + 255) / 256) : 0;
    hipLaunchKernelGGL(sep_table_kernel, dim3((unsigned)(kSepTableBlocks + kSepStatG + gcols)), dim3(256), 0, s, a);
    const int64_t kt = (a.K + 31) / 32, ot = (a.O + 127) / 128;
    const int64_t x_blocks = a.need_w ? kt * ((a.M + 127) / 128) : 0, w_blocks = kt * ot, g_blocks = ot * ((a.M + 31) / 32);
    const int64_t expand = x_blocks + w_blocks + g_blocks;
    hipLaunchKernelGGL(sep_expand_bwd_kernel, dim3((unsigned)std::max<int64_t>(expand, kPrepBlocksX + kPrepBlocksW)),
                       dim3(256), 0, s, a, (int)x_blocks, (int)w_blocks, prep);
    return hipGetLastError();
}

// The backward's products, into the dX and dVth planes.
hipError_t sep_backward_products(const SepPlan& p, SepArgs a, char* ws, hipStream_t s) {
    sep_point_backward(p, a, ws);
    SepGemm g{};
    g.head = a.head;
    g.M = a.M;
    g.K = a.K;
    g.O = a.O;
    g.Kp = p.Kp;
    g.Op = p.Op;
    g.xscale = a.xscale;
    g.gscale = a.gscale;
    g.gscaleT = a.gscaleT;
    g.x = a.x;
    g.in_affine = a.in_affine;
    g.in_lo = a.in_lo;
    g.in_hi = a.in_hi;
    g.tab2 = a.tab2;
    g.tabE = a.tabE;
    g.tT = a.tT;
    g.dv_all = a.lut_n > 0 ? 0 : 1;
    const int64_t tile = p.big ? 256 : 128;
    int64_t blocks = 0;
    auto add = [&](int kind, const _Float16* x, const _Float16* y, int64_t b_rows, int64_t inner, int split, float*& out,
                   int64_t plane, int rows) {  // rows: of an input, at most
        if (split < 1) return;
        g.p[g.n++] = SepProduct{reinterpret_cast<const char*>(x), reinterpret_cast<const char*>(y), kind, a.K, b_rows,
                                inner, split, out};
        out += split * plane;
        blocks += ((a.K + 1) / 2 * 2 * rows + tile - 1) / tile * ((b_rows + tile - 1) / tile) * split;
    };
    float* dx = reinterpret_cast<float*>(ws + p.off_planes);
    float* dv = reinterpret_cast<float*>(ws + p.off_planes_dv);
    const int64_t px = a.M * a.K, pv = 2 * p.Kp * p.Op;
    const int R = p.max_terms;
    if (a.need_x) add(kSepDx, a.wop, a.gop, a.M, a.O, p.split_dx, dx, px, R / 2);
    if (a.need_w) add(kSepDv, a.xop, a.gopT, a.O, a.M, p.split_dv, dv, pv, g.dv_all ? R : R / 2);
    if (a.need_x) add(kSepDxUpper, a.wops, a.goph, a.M, a.O, p.split_dxs, dx, px, R / 2);
    if (a.need_w) add(kSepDvUpper, a.xops, a.gophT, a.O, a.M, p.split_dvs, dv, pv, R / 2);
    if (a.need_x) add(kSepDxHarm, a.woph, a.goph, a.M, a.O, p.split_dxh, dx, px, R);
    if (a.need_w) add(kSepDvHarm, a.xoph, a.gophT, a.O, a.M, p.split_dvh, dv, pv, R);
    launch_sep_gemm<false>(p.big, (unsigned)blocks, g, s);
    return hipGetLastError();
}
