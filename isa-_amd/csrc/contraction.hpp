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
// of the branches.
//
// Precision. The coefficients grow by 2^50 and more from the lowest inputs to the highest ones, and which of them
// count is G's and the thresholds' affair: the highest tokens may carry no gradient, the highest inputs may
// have equal thresholds. So operands are kept to a relative precision, with fp32's exponents: as a sum of
// bf16, three for the first terms (24 bits; six products a pair of operands: all but those below 2^-24),
// two for the next (16 bits, three products), one for the last, whose coefficients are below 9e-2 and 4e-5
// of the first one's. At 8 terms 2, 4 and 2 (dVth, whose first term has no counterpart in a difference, 4, 2
// and 2): 26 (32) products per cell where the cell itself costs 32 (forward) or 52 (backward) VALU
// instructions, four or eight of them transcendental; at 16 terms 52 (64). Only powers of two common to a
// whole operand are taken out. The differences T_j(t+) - T_j(t-) are formed in fp64 before they are
// rounded, so that a cell does not lose the bits in which its two branches agree; equal thresholds give zero.
// c_j, d_j and g_j come from tables over x built per call in fp64 (cubic interpolation, step at most
// kSepStep of 2 n U_T: 2e-8 relative; the step is a power of two, so that a position within a step is exact
// in fp32). Emulated in float64, rows at one input: 2.6e-7 of the output's own scale forward, 3e-7 dVth.
//
// Measured (formula, 768 x 3072 at 2048 tokens, initial thresholds, R = 8): forward 4.29 ms by the per-cell
// kernels, 0.32 ms here; backward 8.17 and 0.85 ms. (Operands as two f16, scaled by row, took 0.22 and
// 0.52 ms, and lost everything 2^-36 below a row's largest value.)
//
// Tables. A lookup is the line between two entries, L(c) = F(c) + S(c) a (1 - a) / 2 with F the
// smooth function through the entries, S its second difference and a the coordinate's fraction
// (the next term is smaller by the relative change from entry to entry, 1.5% at 4096 entries).
// With a (1 - a) = 1/6 - sum_q cos(2 pi q a) / (pi q)^2 and c = xs - ws,
//     L(xs - ws) = (F + S / 12)(xs - ws)
//                  - sum_q S(xs - ws) (cos 2 pi q xs cos 2 pi q ws + sin 2 pi q xs sin 2 pi q ws) / (2 pi^2 q^2):
// the first part is smooth and expands as above, the others are 1e-4 of it. S falls with the threshold as the
// current does where the transistor is in weak inversion (there the kinks count most), more slowly or not at
// all above: it is a combination of two exponentials in t, fitted per point of the x table (what they leave
// is 2e-6 of a current's difference, 5e-6 of a slope's). So a harmonic is four values per input, one bf16
// each. As many harmonics are summed as leave less than the per-cell kernels round, row by row: four at 4096
// entries, two at 8192, one at 16384. Errors of a row's own scale, all inputs of it at one voltage, the largest
// over -1 to 3.8 V, per-cell kernels against this: 4096 entries forward 6.9e-6 and 3.6e-6, dX 1.5e-5 and
// 1.2e-5, dVth 5.0e-6 and 2.1e-6; 8192 entries 6.9e-6 and 2.1e-6, 1.9e-5 and 7.4e-6, 5.1e-6 and 1.3e-6; over
// 1.06 V at 8192 entries 4.5e-6 and 1.2e-6, 4.7e-6 and 1.7e-6, 5.0e-6 and 1.2e-6. 768 x 3072 at 8192 tokens,
// forward / backward, per-cell kernels against this: 4096 entries 4.35 / 8.65 ms and 1.68 / 4.05, 8192 entries
// 4.69 / 9.32 and 1.37 / 3.47; over 1 V the forward at 4096 entries 4.58 and 2.60. Sums of T's
// differences give back the entries exactly. A table that is not smooth (bf16 entries) runs the
// per-cell kernels.
//
// R is chosen per call on the device from the thresholds' spread (sep_terms); a call whose
// operands do not suit (non-finite values, x near -V_sat or spread over more than the table
// holds, thresholds spread too far) runs the per-cell kernels, which return at once otherwise.

typedef __bf16 sep_b8 __attribute__((ext_vector_type(8)));
typedef __bf16 sep_b4 __attribute__((ext_vector_type(4)));
typedef __bf16 sep_b2 __attribute__((ext_vector_type(2)));
typedef float sep_f16 __attribute__((ext_vector_type(16)));

constexpr int kSepStatX = 1024, kSepStatW = 256;  // blocks of the ranges of x and of the thresholds
constexpr int kSepStatG = 512;          // blocks of the largest |G|
constexpr int kSepGridMax = 16384;      // x-table points, at most
constexpr double kSepStep = 0.0148;     // x-table step in units of 2 n U_T
constexpr int kSepMaxTerms = 16;
constexpr int kSepLutMin = 4000, kSepLutMax = 65536;  // table entries: the kinks small enough, a thread per partial
constexpr int kSepMaxHarmonics = 4;

// Widest threshold spread, in units of 2 n U_T, that R = 8 and 16 terms take: there the
// truncation is 2e-7 of the gradients (the forward's is ten times smaller). More would converge
// (16 terms to 4.4), but as the spread grows the per-cell kernels lose fewer bits to the branches'
// difference while the sums here have more terms. Own scales, tokens of all magnitudes, 192 x 768 at 3700
// tokens: 0.2142 V forward 2.7e-7, dX 4.3e-7, dVth 2.1e-7; 0.3 V 1.9e-7, 2.0e-7, 1.8e-7.
__host__ __device__ inline int sep_terms(float spread_u) { return spread_u <= 1.12f ? 8 : spread_u <= 1.45f ? 16 : 0; }

// Table calls. Two functions a harmonic fit the currents' second differences to 2e-6 of a lookup's
// difference over spreads up to 5 units, the slopes' to 5e-6 up to 1.12 units and, as growth^2, to what
// the per-cell kernels round (2.5e-6) over wider ones where entries grow by at most 2.06%.
__host__ __device__ inline int sep_terms_lut(float spread_u, float growth, bool backward) {
    return spread_u <= 1.12f ? 8 : spread_u <= 5.0f && !(backward && growth > 0.0206f) ? 16 : 0;
}
constexpr int kSepLutWideMin = 6000;  // entries that grow by 2.06% over the transistor's 13 V: operands for 16 terms

// What the passes of a call share, in its workspace.
struct SepHead {
    int took;     // for the caller: 1 where the contraction took the call
    int terms;    // 0: the per-cell kernels run
    unsigned gmax;  // backward: bits of the largest |G|: not finite: the per-cell kernels run
    int rough;    // 1: the series does not converge as its terms assume, 2: a sample of the thresholds or of
                  // the table ruled the contraction out (then the other fields are not set): the per-cell kernels run
    int harmonics;  // of the table's kinks that are summed: 0, 1, 2 or 4
    int n_grid;
    float xlo, xhi, wlo, whi;
    float lut_min, lut_scale;  // table coordinate (v - lut_min) * lut_scale
    float x0, step, inv_step; // table point i stands for x0 + i * step; step a power of two, x0 a multiple of it
    double wc, inv_wh, wh;   // t = (w - wc) * inv_wh
    float gw, gu;             // second differences are combinations of exp(gw t) and exp(gu t)
    float scale, inv_scale;   // of the x tables, a power of two: the largest current is near 2^60
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
    float4* lut_info;        // per 256 entries {largest relative change from entry to entry, 1 where they do not suit, largest |entry|, 0}
    float* tabE;             // second difference's coefficients, -r e_i / (2 pi^2), scaled: [n_grid][2]
    // workspace
    SepHead* head;
    float2* xpart;           // [kSepStatX]
    float2* wpart;           // [kSepStatW]
    float* tab;              // forward c_j r (j = 1..R), backward d_j r (j = 0..R-1), scaled: [n_grid][R]
    float* tab2;             // backward g_j (j = 1..R)
    char* xop;               // forward [M] rows
    char* wop;               // forward [O] rows
    // backward, by parts {singles, pairs, triples} and the harmonics: rows of inputs and terms
    char* xcls[4];           // over the tokens
    char* wcls[4];           // over the outputs
    char* gop;               // triples: [M] rows over the outputs
    char* gops;              // singles
    char* gopT;              // triples: [O] rows over the tokens
    char* gopTs;             // singles
    float2* tT;              // backward [K][Op]: {t+, t-}
    int64_t Op;
    int need_x, need_w;
};

__device__ inline float sep_input(const SepArgs& a, float x, float s, float b) {
    return a.in_affine ? input_map(x, s, b, a.in_lo, a.in_hi) : x;
}

// Layouts. An operand's values are kept as one, two or three bf16 (the value, what rounding it left,
// what rounding that left), in runs of 16 inner elements: all first parts, then the second parts, then
// the third ones, 32 bytes each. The matrix kernel reads an operand's row in slabs of up to 128 bytes:
// 64 singles, 32 pairs, 16 triples.
// Forward, a row's inner elements: the singles (the last terms, then the harmonics), the pairs and the
// triples (the first terms): the small terms are summed first. Inputs are padded to 32. Terms are
// ordered (term / 4, input, term % 4), where a class has two (input, term).
// Backward, tokens or outputs inside, padded to 64, an operand per class; rows in blocks of eight: four
// terms of an even input and of the odd one after it, or where a class has two terms those of two inputs
// and of the next two, so that a lane of the matrix cores' result holds whole inputs.
// Harmonics: an input has four values for each, two coefficients times its cosine, two times its sine.
struct SepClasses {
    int n3, n2, n1;  // terms kept as triples, pairs and singles, in this order
    __host__ __device__ constexpr int first(int parts) const { return parts == 3 ? 0 : parts == 2 ? n3 : n3 + n2; }
    __host__ __device__ constexpr int count(int parts) const { return parts == 3 ? n3 : parts == 2 ? n2 : n1; }
};
// The forward's and dX's terms, and dVth's (whose first one, j = 0, has no counterpart in a difference).
__host__ __device__ constexpr SepClasses sep_classes(int terms, bool dv) {
    return terms == 8 ? (dv ? SepClasses{4, 2, 2} : SepClasses{2, 4, 2}) : (dv ? SepClasses{8, 4, 4} : SepClasses{4, 8, 4});
}
__host__ __device__ inline int64_t sep_inputs(int64_t K) { return (K + 31) / 32 * 32; }
__host__ __device__ inline int64_t sep_inner(int64_t n) { return (n + 63) / 64 * 64; }
// Byte offsets of the parts of a forward row, and its bytes.
struct SepRow {
    int64_t harm, pairs, triples, bytes;
    __host__ __device__ SepRow(int64_t K, int terms, int harmonics) {
        const SepClasses c = sep_classes(terms, false);
        const int64_t kc = sep_inputs(K);
        harm = kc * c.n1 * 2;
        pairs = harm + kc * harmonics * 8;
        triples = pairs + kc * c.n2 * 4;
        bytes = triples + kc * c.n3 * 6;
    }
};
// Row of input k's value v of its `count` among a backward class's rows; the rows that hold K inputs.
__host__ __device__ inline int64_t sep_row(int64_t k, int count, int v) {
    return count == 2 ? (k >> 2) * 8 + (k & 3) * 2 + v
                      : ((k >> 1) * (count / 4) + (v >> 2)) * 8 + (k & 1) * 4 + (v & 3);
}
__host__ __device__ inline int64_t sep_rows(int64_t K, int count) {
    return count == 2 ? (K + 3) / 4 * 8 : (K + 1) / 2 * 2 * count;
}

// ----------------------------------------------------------------------------------
// Statistics: ranges of x and of the thresholds, and the largest |G|. NaN makes a range infinite
// and a maximum non-finite. HBM-bound: x, the thresholds and G are read once.
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
// sums those before its range itself), as the smooth part F + S / 12 and S, how fast they change (up or
// down, or by their curvature: it sets the x table's step, the terms and the harmonics), and whether they
// suit: fourth differences within 3e-6 of the entries (what the cubic interpolation and the two
// terms of the lookup's line leave out), and for the backward a slope table that is the current
// table's slope (dX takes the currents from it; within 2e-5 of the difference).
__device__ inline void sep_lut_block(const SepArgs& a, int b) {
    constexpr int kHalo = 2, kSpan = 256 + 2 * kHalo;
    __shared__ double s_t[kSpan];
    __shared__ double s_sum[4];
    __shared__ float s_growth[4], s_big[4];
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
        const double least = fmin(fabs(v), fabs(p1));
        if (least > 1e-30) growth = fmaxf((float)(fabs(p1 - v) / least), sqrtf((float)(fabs(second) / fabs(v))));
        if (v * p1 < 0.0) bad = true;
        if (bwd) {  // the current's difference against the slope's integral (error of fourth order)
            const double di = (double)r0[(size_t)j * 4 + 1];
            const double want = (0.5 * (v + p1) - ((p2 - p1) - (v - m1)) / 24.0) / a.lut_scale;
            const double cur = fabs((double)r0[(size_t)j * 4] + (double)(j + kPad) * di);
            if (!(fabs(di - want) <= 2e-5 * fabs(want) + 4e-7 * cur + 1e-42)) bad = true;
        }
    }
    if (j < n) a.lut_val[j] = make_double2(s_t[i] + second / 12.0, second);
    if (bad) atomicOr(&s_bad, 1);
    float big = j < n ? fabsf((float)s_t[i]) : 0.0f;
    for (int d = 32; d > 0; d >>= 1) {
        growth = fmaxf(growth, __shfl_xor(growth, d));
        big = fmaxf(big, __shfl_xor(big, d));
    }
    if ((t & 63) == 0) {
        s_growth[t >> 6] = growth;
        s_big[t >> 6] = big;
    }
    __syncthreads();
    if (t == 0)
        a.lut_info[b] = make_float4(fmaxf(fmaxf(s_growth[0], s_growth[1]), fmaxf(s_growth[2], s_growth[3])), (float)s_bad,
                                    fmaxf(fmaxf(s_big[0], s_big[1]), fmaxf(s_big[2], s_big[3])), 0.0f);
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
    float growth_all = 0.0f;
    bool bad = false;
    if (a.lut_n > 0) {
        const bool bwd = a.tab2 != nullptr;  // entries {A, dT}, backward the slope table's
        const int i = 2 + (int)((int64_t)place * (a.lut_n - 6) / 16);
        const float2 r = *reinterpret_cast<const float2*>(a.lut + (size_t)(kPad + i - 2 + off) * (bwd ? 4 : 2) + (bwd ? 2 : 0));
        const double d0 = __shfl(r.y, place * 4), d1 = __shfl(r.y, place * 4 + 1), d2 = __shfl(r.y, place * 4 + 2),
                     d3 = __shfl(r.y, place * 4 + 3);
        const double v = (double)__shfl(r.x, place * 4 + 2) + (double)(i + kPad) * d2;  // entry i, to 1e-5
        bad = !(fabs((d3 - d0) - 3.0 * (d2 - d1)) <= 4e-6 * fabs(v) + 2e-42);
        float growth = fabs(v) > 1e-30 ? (float)fabs(d2 / v) : 0.0f;  // (at most the whole table's)
        for (int d = 32; d > 0; d >>= 1) growth = fmaxf(growth, __shfl_xor(growth, d));
        growth_all = 0.999f * growth;
        ua = 0.5 * (double)growth_all * a.lut_scale;
    }
    sep_minmax(wp, lo, hi);
    sep_minmax(wn, lo, hi);
    sep_wave_minmax(lo, hi);
    const float spread = (float)(((double)hi - (double)lo) * ua);
    const int terms = a.lut_n > 0 ? sep_terms_lut(spread, growth_all, a.tab2 != nullptr) : sep_terms(spread);
    return __builtin_amdgcn_readfirstlane((int)(__any(bad) || terms == 0 || terms > a.max_terms)) != 0;
}

// Blocks: kSepStatX of x, kSepStatW of the thresholds, ceil(lut_n / 256) of the table, then the
// layer glue's gradient blocks (glue.geff).
__global__ __launch_bounds__(256) void sep_stat_kernel(SepArgs a, PrepArgs prep, GlueGradArgs glue) {
    int b = blockIdx.x;
    const int t = threadIdx.x;
    const float as = a.in_affine ? a.in_affine[0] : 1.0f, ab = a.in_affine ? a.in_affine[1] : 0.0f;
    const int lut_blocks = (a.lut_n + 255) / 256;
    if (b < kSepStatX + kSepStatW + lut_blocks) {
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
        const int64_t n = a.M * a.K, stride = (int64_t)kSepStatX * 256;
        for (int64_t e = (int64_t)b * 256 + t; e < n; e += 4 * stride) {
            float v[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) v[q] = a.x[e + q * stride < n ? e + q * stride : e];
#pragma unroll
            for (int q = 0; q < 4; ++q) sep_minmax(sep_input(a, v[q], as, ab), lo, hi);
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
    glue_grad_block(glue, b % kGlueBlocks, b / kGlueBlocks, (int)(glue.Op / 256));
}

// The largest |G| (blocks of the table kernel's launch, a wave per row of G).
__device__ inline void sep_grad_block(const SepArgs& a, int b) {
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    unsigned all = 0;
    for (int64_t m = (int64_t)b * 4 + wave; m < a.M; m += (int64_t)kSepStatG * 4) {
        const float* row = a.g + m * a.ldg;
        for (int64_t o = lane; o < a.O; o += 256) {
            unsigned v[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) v[q] = sep_bits(row[o + q * 64 < a.O ? o + q * 64 : o]);
            all = max(all, max(max(v[0], v[1]), max(v[2], v[3])));
        }
    }
    for (int d = 32; d > 0; d >>= 1) all = max(all, (unsigned)__shfl_xor((int)all, d));
    __shared__ unsigned s_all;  // one atomic per block: they all meet at one address
    if (t == 0) s_all = 0;
    __syncthreads();
    if (lane == 0) atomicMax(&s_all, all);
    __syncthreads();
    if (t == 0) atomicMax(&a.head->gmax, s_all);
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

// Blocks: kSepTableBlocks of the tables, then (backward) kSepStatG of G.
__global__ __launch_bounds__(256) void sep_table_kernel(SepArgs a) {
    __shared__ float2 s_x, s_w, s_info, s_big;
    __shared__ SepHead s_head;
    __shared__ double s_cos[4 * kSepMaxTerms], s_val[256], s_sec[256], s_d[256], s_fit[4][kSepMaxTerms];
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
        const float4 info = t * 256 < a.lut_n ? a.lut_info[t] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        block_minmax(lo, hi, &s_x);
        __syncthreads();
        block_minmax(w.x, w.y, &s_w);
        __syncthreads();
        block_minmax(-info.y, info.x, &s_info);  // (-1 where some do not suit, growth)
        __syncthreads();
        block_minmax(0.0f, info.z, &s_big);
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
        const int terms = lut ? sep_terms_lut(spread, (float)growth, a.tab2 != nullptr) : sep_terms(spread);
        bool ok = finite && terms > 0 && terms <= a.max_terms && rlo > 0.1 && rhi > 0.1 &&
                  points <= (double)kSepGridMax && fmax(fabs((double)xlo), fabs((double)xhi)) < step * (1 << 23);
        if (lut) {  // every lookup inside the table, the x table's margin included
            // root mean square of the harmonics left out, in records: 0.0373 growth without any, 0.0103
            // after one, 0.0050 after two, 0.0021 after four; the per-cell kernels round to about 1e-4
            const double left = 7.7e-5;
            h.harmonics = 0.0373 * growth <= left ? 0 : 0.0103 * growth <= left ? 1 : 0.0050 * growth <= left ? 2 : 4;
            const double margin = 4.0 * step * a.lut_scale + 4.0;
            // (four to 3.1%: past it pairs of close thresholds far below threshold, where the per-cell
            // kernels' coordinates are exact to 2^-14 of a record, are further off: 3600 entries 1.4 times)
            ok = ok && s_info.x == 0.0f && growth > 1e-6 && growth <= 0.031 &&
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
            // below threshold they fall with the threshold as the current does; above it the currents' as
            // its root, the slopes' rise. (Narrow spreads: exponents far enough apart to be told apart.)
            h.gw = lut ? -fmaxf((float)(log1p(growth) * a.lut_scale * h.wh), 0.25f) : 0.0f;
            h.gu = a.tab2 ? -0.5f * h.gw : 0.5f * h.gw;
            int e = 60;
            if (lut && s_big.y > 0.0f) e = max(-120, min(120, 60 - ilogbf(s_big.y)));
            h.scale = ldexpf(1.0f, e);
            h.inv_scale = ldexpf(1.0f, -e);
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
            g->gw = h.gw;
            g->gu = h.gu;
            g->scale = h.scale;
            g->inv_scale = h.inv_scale;
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
    if (h.harmonics > 0) {  // least squares over the Chebyshev points: e = s_fit[0..1] S, of s_fit[2..3]
        __syncthreads();
        if (t < R) {
            s_fit[2][t] = exp((double)h.gw * s_cos[2 * t + 1]);
            s_fit[3][t] = exp((double)h.gu * s_cos[2 * t + 1]);
        }
        __syncthreads();
        if (t < R) {
            double aa = 0.0, ab = 0.0, bb = 0.0;
            for (int q = 0; q < R; ++q) {
                aa += s_fit[2][q] * s_fit[2][q];
                ab += s_fit[2][q] * s_fit[3][q];
                bb += s_fit[3][q] * s_fit[3][q];
            }
            const double det = aa * bb - ab * ab;
            s_fit[0][t] = (bb * s_fit[2][t] - ab * s_fit[3][t]) / det;
            s_fit[1][t] = (aa * s_fit[3][t] - ab * s_fit[2][t]) / det;
        }
    }
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
        if (h.harmonics > 0 && n < 2)
            for (int q = 0; q < R; ++q) e2 += s_sec[pl * R + q] * s_fit[n][q];
        __syncthreads();
        if (i0 + pl < h.n_grid) {
            const size_t e = (size_t)(i0 + pl) * R + n;
            if (direct) {
                a.tab[e] = (float)(d * r * (double)h.scale);
            } else {  // c_j from d_(j-1) = d and d_(j+1)
                const double d_next = j < R ? s_d[t + 1] : 0.0, d_after = j + 1 < R ? s_d[t + 2] : 0.0;
                const double c = -h.wh / (2.0 * j) * (d - d_after);
                if (a.tab2) {
                    a.tab[e] = (float)((n == 0 ? 0.5 * d : d) * r * (double)h.scale);
                    a.tab2[e] = (float)(r * (d_next - r / a.v_sat * c));
                } else {
                    a.tab[e] = (float)(c * r * (double)h.scale);
                }
            }
            if (h.harmonics > 0 && n < 2)
                a.tabE[(size_t)(i0 + pl) * 2 + n] = (float)(-r * e2 * 0.050660591821168886 * (double)h.scale);  // 1 / (2 pi^2)
            // the last coefficients of a table that grows otherwise than its steepest part says
            if (lut && n == 0) {
                const int last = direct ? R - 2 : R - 1;  // of degree R - 1
                double big = 0.0;
                for (int q = direct ? 0 : 1; q < R; ++q) big = fmax(big, fabs(s_d[t + q]));
                const double mean = direct ? 0.0 : fabs(0.5 * s_d[t]);
                if (!(fabs(s_d[t + last]) <= 1e-5 * big + 1e-6 * mean + 1e-35)) atomicOr(&a.head->rough, 1);
            }
            // or second differences that the two functions do not fit
            if (h.harmonics > 0 && n == 2) {
                double big = 0.0, e0 = 0.0, e1 = 0.0, left = 0.0;
                for (int q = 0; q < R; ++q) {
                    e0 += s_sec[pl * R + q] * s_fit[0][q];
                    e1 += s_sec[pl * R + q] * s_fit[1][q];
                }
                for (int q = 0; q < R; ++q) {
                    const double u = s_sec[pl * R + q] - e0 * s_fit[2][q] - e1 * s_fit[3][q];
                    left += u * u;
                }
                for (int q = direct ? 0 : 1; q < R; ++q) big = fmax(big, fabs(s_d[t - 2 + q]));
                const double mean = direct ? 0.0 : fabs(0.5 * s_d[t - 2]);
                if (!(0.05 * sqrt(left / R) <= 1e-5 * big + 1e-6 * mean + 1e-35)) atomicOr(&a.head->rough, 1);
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

// Four coefficients from the even j on (8-byte aligned: a class may begin at term 2).
__device__ inline float4 sep_eval4(const float* tab, int R, const SepAt& at, int j) {
    typedef float four __attribute__((ext_vector_type(4), aligned(8)));
    const float* p = tab + (size_t)at.i * R + j;
    const four v0 = *reinterpret_cast<const four*>(p), v1 = *reinterpret_cast<const four*>(p + R);
    const four v2 = *reinterpret_cast<const four*>(p + 2 * R), v3 = *reinterpret_cast<const four*>(p + 3 * R);
    float4 s;
    s.x = fmaf(at.w[3], v3.x, fmaf(at.w[2], v2.x, fmaf(at.w[1], v1.x, at.w[0] * v0.x)));
    s.y = fmaf(at.w[3], v3.y, fmaf(at.w[2], v2.y, fmaf(at.w[1], v1.y, at.w[0] * v0.y)));
    s.z = fmaf(at.w[3], v3.z, fmaf(at.w[2], v2.z, fmaf(at.w[1], v1.z, at.w[0] * v0.z)));
    s.w = fmaf(at.w[3], v3.w, fmaf(at.w[2], v2.w, fmaf(at.w[1], v1.w, at.w[0] * v0.w)));
    return s;
}

__device__ inline float2 sep_eval2(const float* tab, int R, const SepAt& at, int j) {
    const float* p = tab + (size_t)at.i * R + j;
    float2 s = make_float2(0.0f, 0.0f);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const float2 v = *reinterpret_cast<const float2*>(p + q * R);
        s.x = fmaf(at.w[q], v.x, s.x);
        s.y = fmaf(at.w[q], v.y, s.y);
    }
    return s;
}

// Stores N neighbouring inner elements (e a multiple of N) of an operand's row as PARTS bf16 each.
template <int N, int PARTS>
__device__ inline void sep_put(char* row, int64_t e, const float* v) {
    typedef __bf16 vec __attribute__((ext_vector_type(N)));
    char* p = row + (e >> 4) * (32 * PARTS) + (e & 15) * 2;
    float rest[N];
#pragma unroll
    for (int q = 0; q < N; ++q) rest[q] = v[q];
#pragma unroll
    for (int part = 0; part < PARTS; ++part) {
        vec w;
#pragma unroll
        for (int q = 0; q < N; ++q) {
            w[q] = (__bf16)rest[q];
            rest[q] -= (float)w[q];
        }
        *reinterpret_cast<vec*>(p + 32 * part) = w;
    }
}

// ----------------------------------------------------------------------------------
// Forward operands: xop[m] = c_j r (a wave per row, lanes along k) and wop[o] = T_j(t+) - T_j(t-).
// HBM-bound.
// ----------------------------------------------------------------------------------

constexpr int kSepExpandBlocks = 2048;

// Walks T_1, T_2, ... of both branches and hands out blocks of four differences.
struct SepChebPair {
    double p0 = 1.0, p1, n0 = 1.0, n1, tp, tn;
    __device__ SepChebPair(double a, double b) : p1(a), n1(b), tp(2.0 * a), tn(2.0 * b) {}
    __device__ void next4(float* v) {  // T_j(t+) - T_j(t-) of the next four j
#pragma clang fp contract(off)  // the same roundings for both branches: equal thresholds give zero
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            v[q] = (float)(p1 - n1);
            const double p2 = tp * p1 - p0, n2 = tn * n1 - n0;
            p0 = p1;
            p1 = p2;
            n0 = n1;
            n1 = n2;
        }
    }
};

// cos and sin of 2 pi q theta, q = 1, 2, ... (theta in revolutions).
struct SepTurn {
    float c1, s1, c, s;
    SepTurn() = default;
    __device__ explicit SepTurn(float theta) {
        const float f = theta - floorf(theta);
        c = c1 = __builtin_amdgcn_cosf(f);
        s = s1 = __builtin_amdgcn_sinf(f);
    }
    __device__ void next() {
#pragma clang fp contract(off)  // the same roundings for both branches of a pair
        const float t = c1 * c - s1 * s;
        s = s1 * c + c1 * s;
        c = t;
    }
};

// 1 / q^2 of harmonic q - 1.
__device__ inline float sep_harm_weight(int q) { return q == 0 ? 1.0f : q == 1 ? 0.25f : q == 2 ? 1.0f / 9.0f : 0.0625f; }

// The nearest table point's two second-difference coefficients (they change by 1.5% from point to
// point, and are 1e-4 of the result).
__device__ inline float2 sep_second(const float* tabE, const SepAt& at) {
    return reinterpret_cast<const float2*>(tabE)[at.i + (at.w[2] > at.w[1] ? 2 : 1)];
}

// A harmonic's four values of an input on the token side (e scaled) ...
__device__ inline void sep_harm_x(float v[4], float2 e, float c, float sn, float weight) {
    v[0] = e.x * c * weight;
    v[1] = e.y * c * weight;
    v[2] = e.x * sn * weight;
    v[3] = e.y * sn * weight;
}

// ... and on the threshold side, differences of the branches' (u: the two functions at t+, t-). Products
// are rounded before they are subtracted, so that equal thresholds give zero.
__device__ inline void sep_harm_w(float v[4], float2 up, float2 un, float cp, float sp, float cn, float sn) {
#pragma clang fp contract(off)
    v[0] = up.x * cp - un.x * cn;
    v[1] = up.y * cp - un.y * cn;
    v[2] = up.x * sp - un.x * sn;
    v[3] = up.y * sp - un.y * sn;
}

__device__ inline float2 sep_kink_functions(const SepHead& h, float t) { return make_float2(expf(h.gw * t), expf(h.gu * t)); }

// Records who takes the call, and clears what its prep would (first block of the operands' launch).
__device__ inline void sep_record(SepHead* head, bool took, const PrepArgs& p) {
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    head->took = took ? 1 : 0;
    if (took && p.stat_bits) *p.stat_bits = 0u;
}

template <int R>
__device__ inline void sep_expand_fwd(const SepArgs& a, const SepHead& h) {
    constexpr SepClasses cls = sep_classes(R, false);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t kc = sep_inputs(a.K);
    const SepRow at_row(a.K, R, h.harmonics);
    const float as = a.in_affine ? a.in_affine[0] : 1.0f, ab = a.in_affine ? a.in_affine[1] : 0.0f;
    // all terms of input k of a row, then its harmonics
    auto terms = [&](char* row, int64_t k, const float* v) {
        sep_put<cls.n3, 3>(row + at_row.triples, k * cls.n3, v);
#pragma unroll
        for (int b = 0; b < cls.n2 / 4; ++b) sep_put<4, 2>(row + at_row.pairs, (b * kc + k) * 4, v + cls.n3 + 4 * b);
        sep_put<cls.n1, 1>(row, k * cls.n1, v + cls.n3 + cls.n2);
    };
    for (int64_t row = (int64_t)blockIdx.x * 4 + wave; row < a.M + a.O; row += (int64_t)gridDim.x * 4) {
        if (row < a.M) {
            char* dst = a.xop + row * at_row.bytes;
            for (int64_t k = lane; k < kc; k += 64) {
                const bool real = k < a.K;
                const float x = sep_input(a, a.x[row * a.K + (real ? k : a.K - 1)], as, ab), one = real ? 1.0f : 0.0f;
                const SepAt at = sep_at(h, x);
                float v[R];
#pragma unroll
                for (int j = 0; j < R; j += 4) {
                    const float4 c = sep_eval4(a.tab, R, at, j);
                    v[j] = c.x * one; v[j + 1] = c.y * one; v[j + 2] = c.z * one; v[j + 3] = c.w * one;
                }
                terms(dst, k, v);
                if (h.harmonics > 0) {
                    const float2 e = sep_second(a.tabE, at);
                    SepTurn turn((x - h.lut_min) * h.lut_scale);
                    for (int q = 0; q < h.harmonics; ++q) {
                        float u[4];
                        sep_harm_x(u, e, turn.c, turn.s, sep_harm_weight(q) * one);
                        sep_put<4, 1>(dst + at_row.harm, (q * kc + k) * 4, u);
                        turn.next();
                    }
                }
            }
        } else {
            const int64_t o = row - a.M;
            char* dst = a.wop + o * at_row.bytes;
            for (int64_t k = lane; k < kc; k += 64) {
                const bool real = k < a.K;  // padded inputs: both branches at the centre
                const double tp = real ? ((double)a.wp[o * a.K + k] - h.wc) * h.inv_wh : 0.0;
                const double tn = real ? ((double)a.wn[o * a.K + k] - h.wc) * h.inv_wh : 0.0;
                SepChebPair c(tp, tn);
                float v[R];
#pragma unroll
                for (int j = 0; j < R; j += 4) c.next4(v + j);
                terms(dst, k, v);
                if (h.harmonics > 0) {
                    const float2 fp = sep_kink_functions(h, (float)tp), fn = sep_kink_functions(h, (float)tn);
                    SepTurn up((float)((h.wc + h.wh * tp) * h.lut_scale)), un((float)((h.wc + h.wh * tn) * h.lut_scale));
                    for (int q = 0; q < h.harmonics; ++q) {
                        float u[4];
                        sep_harm_w(u, fp, fn, up.c, up.s, un.c, un.s);
                        sep_put<4, 1>(dst + at_row.harm, (q * kc + k) * 4, u);
                        up.next();
                        un.next();
                    }
                }
            }
        }
    }
}

// Where the per-cell kernels take the call: their prep, in the same launch (unless the statistics'
// launch has run it).
__global__ __launch_bounds__(256) void sep_expand_fwd_kernel(SepArgs a, PrepArgs prep) {
    const bool takes = sep_takes(a.head);
    sep_record(a.head, takes, prep);
    if (!takes) {
        if (blockIdx.x < kPrepBlocksX + kPrepBlocksW && a.head->rough != 2) prep_block(prep, blockIdx.x);
        return;
    }
    const SepHead h = *a.head;
    if (h.terms == 8)
        sep_expand_fwd<8>(a, h);
    else
        sep_expand_fwd<16>(a, h);
}

// ----------------------------------------------------------------------------------
// Backward operands, tokens or outputs inside: the rows (input, term) of d_j r over the tokens and of
// T_j(t+) - T_j(t-) over the outputs, with tT[k][o] = {t+, t-}, and G in both directions, scaled by a
// power of two to at most 1. Tiles of 32 inputs (or rows of G) by 128 inner elements go through LDS, so
// that reads run along the tensors' rows and writes along the inner index, four elements a thread.
// HBM-bound.
// ----------------------------------------------------------------------------------

constexpr int kSepTilePitch = 132;

// Four inner elements from e on of class PARTS' rows of input k: v[term][element].
template <int R, bool DV, int PARTS>
__device__ inline void sep_put_rows(char* op, int64_t inner, int64_t k, int64_t e, const float (*v)[4]) {
    constexpr SepClasses cls = sep_classes(R, DV);
    constexpr int first = cls.first(PARTS), count = cls.count(PARTS);
    char* row = op + sep_row(k, count, 0) * inner * (2 * PARTS);
#pragma unroll
    for (int i = 0; i < count; ++i)
        sep_put<4, PARTS>(row + (sep_row(0, count, i) - sep_row(0, count, 0)) * inner * (2 * PARTS), e, v[first + i]);
}

template <int R>
__device__ inline void sep_expand_tokens(const SepArgs& a, const SepHead& h, int b, float (*s_x)[kSepTilePitch]) {
    const int t = threadIdx.x, n_mt = (int)((a.M + 127) / 128);
    const int64_t inner = sep_inner(a.M), m0 = (int64_t)(b % n_mt) * 128, k0 = (int64_t)(b / n_mt) * 32;
    const float as = a.in_affine ? a.in_affine[0] : 1.0f, ab = a.in_affine ? a.in_affine[1] : 0.0f;
    for (int q = t; q < 32 * 128; q += 256) {
        const int64_t m = m0 + (q >> 5), k = k0 + (q & 31);
        s_x[q & 31][q >> 5] = m < a.M && k < a.K ? sep_input(a, a.x[m * a.K + k], as, ab) : h.xlo;
    }
    __syncthreads();
    for (int q = t; q < 32 * 32; q += 256) {
        const int64_t k = k0 + (q >> 5), m = m0 + 4 * (q & 31);
        if (k >= a.K || m >= inner) continue;
        const float4 x4 = *reinterpret_cast<const float4*>(&s_x[q >> 5][4 * (q & 31)]);
        const float x[4] = {x4.x, x4.y, x4.z, x4.w};
        float v[R][4];
        SepAt at[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            at[i] = sep_at(h, x[i]);
            const float one = m + i < a.M ? 1.0f : 0.0f;
#pragma unroll
            for (int j = 0; j < R; j += 4) {
                const float4 u = sep_eval4(a.tab, R, at[i], j);
                v[j][i] = u.x * one; v[j + 1][i] = u.y * one; v[j + 2][i] = u.z * one; v[j + 3][i] = u.w * one;
            }
        }
        sep_put_rows<R, true, 3>(a.xcls[2], inner, k, m, v);
        sep_put_rows<R, true, 2>(a.xcls[1], inner, k, m, v);
        sep_put_rows<R, true, 1>(a.xcls[0], inner, k, m, v);
        if (h.harmonics > 0) {
            SepTurn turn[4];
            float2 e[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                e[i] = sep_second(a.tabE, at[i]);
                if (m + i >= a.M) e[i] = make_float2(0.0f, 0.0f);
                turn[i] = SepTurn((x[i] - h.lut_min) * h.lut_scale);
            }
            for (int qh = 0; qh < h.harmonics; ++qh) {
                const float weight = sep_harm_weight(qh);
                float w[4][4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float u[4];
                    sep_harm_x(u, e[i], turn[i].c, turn[i].s, weight);
                    turn[i].next();
#pragma unroll
                    for (int j = 0; j < 4; ++j) w[j][i] = u[j];
                }
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    sep_put<4, 1>(a.xcls[3] + sep_row(k, 4 * h.harmonics, 4 * qh + j) * inner * 2, m, w[j]);
            }
        }
    }
}

template <int R>
__device__ inline void sep_expand_thresholds(const SepArgs& a, const SepHead& h, int b, float (*s_p)[kSepTilePitch],
                                             float (*s_n)[kSepTilePitch]) {
    const int t = threadIdx.x, n_ot = (int)((a.O + 127) / 128);
    const int64_t inner = sep_inner(a.O), o0 = (int64_t)(b % n_ot) * 128, k0 = (int64_t)(b / n_ot) * 32;
    // padded outputs: both branches near the centre, so that their differences vanish
    for (int q = t; q < 32 * 128; q += 256) {
        const int64_t o = o0 + (q >> 5), k = k0 + (q & 31);
        const bool real = o < a.O && k < a.K;
        s_p[q & 31][q >> 5] = real ? a.wp[o * a.K + k] : (float)h.wc;
        s_n[q & 31][q >> 5] = real ? a.wn[o * a.K + k] : (float)h.wc;
    }
    __syncthreads();
    for (int q = t; q < 32 * 32; q += 256) {
        const int64_t k = k0 + (q >> 5), o = o0 + 4 * (q & 31);
        if (k >= a.K || o >= inner) continue;
        const float* wp = &s_p[q >> 5][4 * (q & 31)];
        const float* wn = &s_n[q >> 5][4 * (q & 31)];
        float tp[4], tn[4], v[R][4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const double p = ((double)wp[i] - h.wc) * h.inv_wh, n = ((double)wn[i] - h.wc) * h.inv_wh;
            tp[i] = (float)p;
            tn[i] = (float)n;
            SepChebPair c(p, n);
            float u[4];
#pragma unroll
            for (int j = 0; j < R; j += 4) {
                c.next4(u);
#pragma unroll
                for (int d = 0; d < 4; ++d) v[j + d][i] = u[d];
            }
        }
        if (a.need_w) {
            float4* dst = reinterpret_cast<float4*>(a.tT + k * a.Op + o);
            dst[0] = make_float4(tp[0], tn[0], tp[1], tn[1]);
            dst[1] = make_float4(tp[2], tn[2], tp[3], tn[3]);
        }
        if (!a.need_x) continue;
        sep_put_rows<R, false, 3>(a.wcls[2], inner, k, o, v);
        sep_put_rows<R, false, 2>(a.wcls[1], inner, k, o, v);
        sep_put_rows<R, false, 1>(a.wcls[0], inner, k, o, v);
        if (h.harmonics > 0) {
            SepTurn up[4], un[4];
            float2 fp[4], fn[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                fp[i] = sep_kink_functions(h, tp[i]);
                fn[i] = sep_kink_functions(h, tn[i]);
                up[i] = SepTurn(wp[i] * h.lut_scale);
                un[i] = SepTurn(wn[i] * h.lut_scale);
            }
            for (int qh = 0; qh < h.harmonics; ++qh) {
                float w[4][4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float u[4];
                    sep_harm_w(u, fp[i], fn[i], up[i].c, up[i].s, un[i].c, un[i].s);
                    up[i].next();
                    un[i].next();
#pragma unroll
                    for (int j = 0; j < 4; ++j) w[j][i] = u[j];
                }
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    sep_put<4, 1>(a.wcls[3] + sep_row(k, 4 * h.harmonics, 4 * qh + j) * inner * 2, o, w[j]);
            }
        }
    }
}

// The power of two that brings |G| to at most 1, and its inverse.
__device__ inline float sep_grad_scale(const SepHead* head, float* inverse) {
    const float big = __uint_as_float(head->gmax);
    int e = big > 0.0f ? -(ilogbf(big) + 1) : 0;
    e = e > 120 ? 120 : e < -120 ? -120 : e;
    *inverse = ldexpf(1.0f, -e);
    return ldexpf(1.0f, e);
}

// G: tiles of 32 rows by 128 outputs.
__device__ inline void sep_expand_grad(const SepArgs& a, int b, float (*s_g)[kSepTilePitch]) {
    const int t = threadIdx.x, n_ot = (int)((a.O + 127) / 128);
    const int64_t mi = sep_inner(a.M), oi = sep_inner(a.O);
    if (b >= n_ot * (int)(mi / 32)) return;  // blocks that only the prep needs
    const int64_t o0 = (int64_t)(b % n_ot) * 128, m0 = (int64_t)(b / n_ot) * 32;
    float inv;
    const float scale = sep_grad_scale(a.head, &inv);
    for (int q = t; q < 32 * 128; q += 256) {
        const int64_t m = m0 + (q >> 7), o = o0 + (q & 127);
        s_g[q >> 7][q & 127] = m < a.M && o < a.O ? a.g[m * a.ldg + o] * scale : 0.0f;
    }
    __syncthreads();
    if (a.need_x) {
        for (int q = t; q < 32 * 32; q += 256) {
            const int64_t m = m0 + (q >> 5), o = o0 + 4 * (q & 31);
            if (m >= a.M || o >= oi) continue;
            const float* v = &s_g[q >> 5][4 * (q & 31)];
            sep_put<4, 3>(a.gop + m * oi * 6, o, v);
            sep_put<4, 1>(a.gops + m * oi * 2, o, v);
        }
    }
    if (a.need_w) {
        for (int q = t; q < 128 * 8; q += 256) {
            const int64_t o = o0 + (q >> 3), m = m0 + 4 * (q & 7);
            if (o >= a.O) continue;
            float v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = s_g[4 * (q & 7) + i][q >> 3];
            sep_put<4, 3>(a.gopT + o * mi * 6, m, v);
            sep_put<4, 1>(a.gopTs + o * mi * 2, m, v);
        }
    }
}

__global__ __launch_bounds__(256, 3) void sep_expand_bwd_kernel(SepArgs a, int x_blocks, int w_blocks, PrepArgs prep) {
    const bool takes = sep_takes(a.head);
    sep_record(a.head, takes, prep);
    if (!takes) {  // the per-cell kernels take the call: their prep
        if (blockIdx.x < kPrepBlocksX + kPrepBlocksW && a.head->rough != 2) prep_block(prep, blockIdx.x);
        return;
    }
    const SepHead h = *a.head;
    __shared__ __align__(16) float s_a[32][kSepTilePitch], s_b[32][kSepTilePitch];
    const int b = blockIdx.x;
    if (b < x_blocks) {
        if (h.terms == 8)
            sep_expand_tokens<8>(a, h, b, s_a);
        else
            sep_expand_tokens<16>(a, h, b, s_a);
    } else if (b < x_blocks + w_blocks) {
        if (h.terms == 8)
            sep_expand_thresholds<8>(a, h, b - x_blocks, s_a, s_b);
        else
            sep_expand_thresholds<16>(a, h, b - x_blocks, s_a, s_b);
    } else {
        sep_expand_grad(a, b - x_blocks - w_blocks, s_a);
    }
}

// ----------------------------------------------------------------------------------
// The product of two operands, C[i][j] = sum_e A[i][e] B[j][e]: tiles of (WM MI 32) x (WN NI 32), one
// slab (up to 128 bytes per row) of both operands at a time in two LDS buffers. A slab holds 64 inner
// elements as singles (one product per pair of fragments), 32 as pairs (three: all but the product of
// the second parts) or 16 as triples (six). A triples' slab is summed by itself, its small products
// first, and added to the sums so far: a sum over 8192 tokens rounds 512 times in place of 3072. A
// slab's loads are issued before the arithmetic of the one before it: 3072 matrix-core cycles per
// 64 KB of operands for the 256 x 256 tile, so that one buffer ahead covers the memory's latency and
// the operands need ~21 bytes per cycle and CU. Rows are 128 bytes of LDS and their eight 16-byte parts
// are stored at part ^ (row / 2 % 8), so that the 16 rows that a quarter-wave reads lie on different
// banks. Rows past the operand's end read its last row (their results are dropped).
// Blocks are dealt so that each XCD works on neighbouring tiles (whose operands its L2 holds).
//
// A launch runs up to eight products after one another in its grid (the backward's dX and dVth, each of
// the triples, the pairs, the singles and the harmonics), so that one's last blocks overlap the next
// one's first.
// ----------------------------------------------------------------------------------

enum SepKind { kSepForward, kSepDx, kSepDv };

struct SepProduct {
    const char* a;
    const char* b;
    int kind;
    int parts;                // backward: of the terms' class; 0: the harmonics
    int64_t a_rows, b_rows;   // dX, dVth: inputs in the place of A's rows
    int64_t inner;            // backward: padded tokens or outputs
    int n_split;
    float* out;               // forward: planes [n_split][M][O]; dX: [n_split][M][K]; dVth: [n_split][2][Kp][Op]
};

struct SepGemm {
    SepProduct p[8];
    int n;
    const SepHead* head;
    int64_t M, K, O, Kp, Op;
    const float* x;
    const float* in_affine;
    float in_lo, in_hi;
    const float* tab2;
    const float* tabE;
    const float2* tT;
};

// T_j(t), T_(j+1)(t) for the first term j of a class or of four in it: 0, 4, 6, 8 or 12
// (T_(a+b) = 2 T_a T_b - T_(a-b)).
__device__ inline float2 sep_cheb_from(int j, float t) {
    if (j == 0) return make_float2(1.0f, t);
    const float t2 = fmaf(2.0f * t, t, -1.0f), t3 = fmaf(2.0f * t, t2, -t);
    const float t4 = fmaf(2.0f * t2, t2, -1.0f), t5 = fmaf(2.0f * t2, t3, -t);
    if (j == 4) return make_float2(t4, t5);
    if (j == 8) return make_float2(fmaf(2.0f * t4, t4, -1.0f), fmaf(2.0f * t4, t5, -t));
    const float t6 = fmaf(2.0f * t3, t3, -1.0f), t7 = fmaf(2.0f * t3, t4, -t);
    if (j == 6) return make_float2(t6, t7);
    return make_float2(fmaf(2.0f * t6, t6, -1.0f), fmaf(2.0f * t6, t7, -t));  // 12
}

// Values of an input in a backward product (0: no such product).
__host__ __device__ inline int sep_values(int kind, int parts, int terms, int harmonics) {
    return parts == 0 ? 4 * harmonics : sep_classes(terms, kind == kSepDv).count(parts);
}

template <int WM, int WN, int MI, int NI, bool FORWARD>
__global__ __launch_bounds__(WM * WN * 64, 2) void sep_gemm_kernel(SepGemm g) {
    constexpr int kThreads = WM * WN * 64, TM = WM * MI * 32, TN = WN * NI * 32;
    constexpr int kLoadA = TM * 8 / kThreads, kLoadB = TN * 8 / kThreads, kRowStep = kThreads / 8;
    extern __shared__ __attribute__((aligned(16))) char s_sep[];
    const SepHead* head = g.head;
    if (!sep_takes(head)) return;
    const int R = __builtin_amdgcn_readfirstlane(head->terms);
    const int harmonics = __builtin_amdgcn_readfirstlane(head->harmonics);
    // the product this block works on: its rows, their bytes, and the slabs of each kind
    int id = blockIdx.x, which = 0, ta = 0, tb = 0, n = 0, values = 0, n1 = 0, n2 = 0, n3 = 0;
    unsigned pitch_a = 0, pitch_b = 0, base2 = 0, base3 = 0;  // (an operand holds less than 4 GiB)
    int64_t a_rows = 0;
    for (;; ++which) {
        if (which >= g.n) return;
        const SepProduct& p = g.p[which];
        if constexpr (FORWARD) {
            const SepRow row(g.K, R, harmonics);
            a_rows = p.a_rows;
            n1 = (int)(row.pairs / 128);
            n2 = (int)((row.triples - row.pairs) / 128);
            n3 = (int)((row.bytes - row.triples) / 96);
            base2 = (unsigned)row.pairs;
            base3 = (unsigned)row.triples;
            pitch_a = pitch_b = (unsigned)row.bytes;
        } else {
            values = sep_values(p.kind, p.parts, R, harmonics);
            a_rows = sep_rows(p.a_rows, values);
            n1 = p.parts <= 1 ? (int)(p.inner / 64) : 0;
            n2 = p.parts == 2 ? (int)(p.inner / 32) : 0;
            n3 = p.parts == 3 ? (int)(p.inner / 16) : 0;
            pitch_a = (unsigned)p.inner * (p.parts == 3 ? 6 : p.parts == 2 ? 4 : 2);
            pitch_b = (unsigned)p.inner * (p.parts >= 2 ? 6 : 2);  // G as pairs: its triples' first parts
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
    const int slabs = n1 + n2 + n3;
    const int s_begin = (int)((int64_t)slabs * split / p.n_split);
    const int s_end = (int)((int64_t)slabs * (split + 1) / p.n_split);

    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wr = wave / WN, wc = wave % WN;
    // this thread's 16 bytes of a slab's rows: where they lie in memory
    const int row0 = t >> 3, part = (t & 7) ^ ((row0 >> 1) & 7);
    const unsigned off = part * 16, off_b2 = FORWARD ? off : (part >> 2) * 96 + (part & 3) * 16;
    const unsigned off3 = (part < 6 ? part : part - 6) * 16;  // (a slab of triples has six)
    constexpr unsigned kStrideB2 = FORWARD ? 128 : 192;
    unsigned pa[kLoadA], pb[kLoadB];
#pragma unroll
    for (int q = 0; q < kLoadA; ++q) {
        const int64_t row = a0 + row0 + q * kRowStep;
        pa[q] = (unsigned)(row < a_rows ? row : a_rows - 1) * pitch_a;
    }
#pragma unroll
    for (int q = 0; q < kLoadB; ++q) {
        const int64_t row = b0 + row0 + q * kRowStep;
        pb[q] = (unsigned)(row < p.b_rows ? row : p.b_rows - 1) * pitch_b;
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
        unsigned ua, ub;
        if (s < n1) {
            ua = ub = (unsigned)s * 128u + off;
        } else if (s < n1 + n2) {
            ua = base2 + (unsigned)(s - n1) * 128u + off;
            ub = base2 + (unsigned)(s - n1) * kStrideB2 + off_b2;
        } else {
            ua = ub = base3 + (unsigned)(s - n1 - n2) * 96u + off3;
        }
        char* dst = s_sep + buf * kBuf + wave * 1024;
#pragma unroll
        for (int q = 0; q < kLoadA; ++q)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(abase + (pa[q] + ua)),
                                             (__attribute__((address_space(3))) void*)(dst + q * kThreads * 16), 16, 0, 0);
#pragma unroll
        for (int q = 0; q < kLoadB; ++q)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(bbase + (pb[q] + ub)),
                                             (__attribute__((address_space(3))) void*)(dst + TM * 128 + q * kThreads * 16), 16, 0, 0);
    };
    auto multiply = [&](const sep_b8* u, const sep_b8* v) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NI; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(u[i], v[j], acc[i][j], 0, 0, 0);
    };
    // 16-byte part `index` (even) + fh of the wave's rows
    auto fragments = [&](const char* base, int index, sep_b8* u, sep_b8* v) {
        const int at = frag ^ (index << 4);
#pragma unroll
        for (int i = 0; i < MI; ++i) u[i] = *reinterpret_cast<const sep_b8*>(base + fa + i * 4096 + at);
#pragma unroll
        for (int j = 0; j < NI; ++j) v[j] = *reinterpret_cast<const sep_b8*>(base + fb + j * 4096 + at);
    };
    if (s_begin < s_end) copy(s_begin, 0);
    int s = s_begin;
    for (const int end = min(s_end, n1); s < end; ++s) {
        const int buf = (s - s_begin) & 1;
        __syncthreads();  // this slab has landed, and the other buffer's has been read
        const char* base = s_sep + buf * kBuf;
        sep_b8 av[4][MI], bv[4][NI];
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) fragments(base, 2 * ks, av[ks], bv[ks]);
        if (s + 1 < s_end) copy(s + 1, buf ^ 1);
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) multiply(av[ks], bv[ks]);
    }
    for (const int end = min(s_end, n1 + n2); s < end; ++s) {
        const int buf = (s - s_begin) & 1;
        __syncthreads();
        const char* base = s_sep + buf * kBuf;
        sep_b8 av[4][MI], bv[4][NI];  // parts 1 and 2 of the first 16 elements, then of the others
#pragma unroll
        for (int q = 0; q < 4; ++q) fragments(base, 2 * q, av[q], bv[q]);
        if (s + 1 < s_end) copy(s + 1, buf ^ 1);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            multiply(av[2 * ks + 1], bv[2 * ks]);
            multiply(av[2 * ks], bv[2 * ks + 1]);
            multiply(av[2 * ks], bv[2 * ks]);
        }
    }
    for (; s < s_end; ++s) {
        const int buf = (s - s_begin) & 1;
        __syncthreads();
        const char* base = s_sep + buf * kBuf;
        sep_b8 av[3][MI], bv[3][NI];
#pragma unroll
        for (int q = 0; q < 3; ++q) fragments(base, 2 * q, av[q], bv[q]);
        if (s + 1 < s_end) copy(s + 1, buf ^ 1);
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            sep_f16 sum[NI] = {};
            auto add = [&](int pa_, int pb_) {
#pragma unroll
                for (int j = 0; j < NI; ++j)
                    sum[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[pa_][i], bv[pb_][j], sum[j], 0, 0, 0);
            };
            add(2, 0);
            add(0, 2);
            add(1, 1);
            add(1, 0);
            add(0, 1);
            add(0, 0);
#pragma unroll
            for (int j = 0; j < NI; ++j) acc[i][j] += sum[j];
        }
    }

    // lane (fl, fh) holds rows q % 4 + 8 (q / 4) + 4 fh of column fl of each 32 x 32 tile
    if constexpr (FORWARD) {
        float* out = p.out + (int64_t)split * g.M * g.O;
        const float inv = head->inv_scale;
#pragma unroll
        for (int i = 0; i < MI; ++i) {
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const int64_t m = a0 + (wr * MI + i) * 32 + (q & 3) + 8 * (q >> 2) + 4 * fh;
                if (m >= g.M) continue;
#pragma unroll
                for (int j = 0; j < NI; ++j) {
                    const int64_t o = b0 + (wc * NI + j) * 32 + fl;
                    if (o < g.O) out[m * g.O + o] = acc[i][j][q] * inv;
                }
            }
        }
    } else {
        const SepHead h = *head;
        // two: a lane's block of four results holds two values of two inputs, otherwise four of one
        const bool harm = p.parts == 0, two = values == 2;
        const int per = two ? 1 : values / 4, sh = __builtin_ctz(per);
        const int first = harm ? 0 : sep_classes(R, p.kind == kSepDv).first(p.parts);
        float inv_g;
        (void)sep_grad_scale(head, &inv_g);
        // keeps the loads of the results that follow from being hoisted: the sums leave few registers
        auto fence = [] { __builtin_amdgcn_sched_barrier(0); };
        // block (i, q) of this wave's rows
        auto block_of = [&](int i, int q) { return (int)(a0 / 8) + (wr * MI + i) * 4 + q; };
        const int K = (int)g.K, M = (int)g.M, O = (int)g.O, Op = (int)g.Op;  // (an operand holds less than 4 GiB)
        if (p.kind == kSepDx) {
            const float as = g.in_affine ? g.in_affine[0] : 1.0f, ab = g.in_affine ? g.in_affine[1] : 0.0f;
            float* out = p.out + (int64_t)split * g.M * g.K;
            const float sc = harm ? inv_g * h.inv_scale : inv_g;
            auto each = [&](auto values_of) {  // values_of(x, block of four in the input) -> their four factors
#pragma unroll
                for (int j = 0; j < NI; ++j) {
                    const int m = (int)b0 + (wc * NI + j) * 32 + fl;
                    const int mc = m < M ? m : M - 1;
                    const float* xrow = g.x + (int64_t)mc * K;
                    float* orow = out + (int64_t)mc * K;
                    float sum = 0.0f;
#pragma unroll
                    for (int i = 0; i < MI; ++i) {
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            const int k = (block_of(i, q) >> sh) * 2 + fh, jb = block_of(i, q) & (per - 1);
                            const float xr = xrow[k < K ? k : K - 1];
                            const float4 v = values_of(g.in_affine ? input_map(xr, as, ab, g.in_lo, g.in_hi) : xr, jb);
                            sum = fmaf(acc[i][j][4 * q], v.x, sum);
                            sum = fmaf(acc[i][j][4 * q + 1], v.y, sum);
                            sum = fmaf(acc[i][j][4 * q + 2], v.z, sum);
                            sum = fmaf(acc[i][j][4 * q + 3], v.w, sum);
                            if (jb == per - 1) {
                                if (m < M && k < K) orow[k] = sum * sc;
                                sum = 0.0f;
                            }
                            fence();
                        }
                    }
                }
            };
            if (harm) {
                each([&](float x, int jb) {
                    const SepAt at = sep_at(h, x);
                    const float th = (x - h.lut_min) * h.lut_scale * (float)(jb + 1);
                    const float f = th - floorf(th), w = sep_harm_weight(jb);
                    const float c = __builtin_amdgcn_cosf(f) * w, sn = __builtin_amdgcn_sinf(f) * w;
                    const float2 e = sep_second(g.tabE, at);
                    return make_float4(e.x * c, e.y * c, e.x * sn, e.y * sn);
                });
            } else if (!two) {
                each([&](float x, int jb) { return sep_eval4(g.tab2, R, sep_at(h, x), first + 4 * jb); });
            } else {
#pragma unroll
                for (int j = 0; j < NI; ++j) {
                    const int m = (int)b0 + (wc * NI + j) * 32 + fl;
                    const int mc = m < M ? m : M - 1;
                    const float* xrow = g.x + (int64_t)mc * K;
                    float* orow = out + (int64_t)mc * K;
#pragma unroll
                    for (int i = 0; i < MI; ++i) {
#pragma unroll
                        for (int q = 0; q < 8; ++q) {
                            const int k = block_of(i, q >> 1) * 4 + 2 * fh + (q & 1);
                            const float xr = xrow[k < K ? k : K - 1];
                            const float x = g.in_affine ? input_map(xr, as, ab, g.in_lo, g.in_hi) : xr;
                            const float2 v = sep_eval2(g.tab2, R, sep_at(h, x), first);
                            if (m < M && k < K)
                                orow[k] = fmaf(acc[i][j][2 * q + 1], v.y, acc[i][j][2 * q] * v.x) * sc;
                            if (q & 1) fence();
                        }
                    }
                }
            }
        } else {
            float* out = p.out + (int64_t)split * 2 * g.Kp * g.Op;
            const float sc = inv_g * h.inv_scale;
            const int64_t branch = g.Kp * Op;
            auto store = [&](int k, int o, float vp, float vn) {
                if (o >= O || k >= K) return;
                float* at = out + (int64_t)k * Op + o;
                at[0] = vp * sc;
                at[branch] = vn * sc;
            };
            if (two) {
#pragma unroll
                for (int j = 0; j < NI; ++j) {
                    const int o = (int)b0 + (wc * NI + j) * 32 + fl, oc = o < O ? o : O - 1;
#pragma unroll
                    for (int i = 0; i < MI; ++i) {
#pragma unroll
                        for (int q = 0; q < 8; ++q) {
                            const int k = block_of(i, q >> 1) * 4 + 2 * fh + (q & 1);
                            const float2 tt = g.tT[(int64_t)(k < K ? k : K - 1) * Op + oc];
                            const float2 up = sep_cheb_from(first, tt.x), un = sep_cheb_from(first, tt.y);
                            store(k, o, fmaf(acc[i][j][2 * q + 1], up.y, acc[i][j][2 * q] * up.x),
                                  fmaf(acc[i][j][2 * q + 1], un.y, acc[i][j][2 * q] * un.x));
                            if (q & 1) fence();
                        }
                    }
                }
                return;
            }
            // share(block of four in the input, their sums, t+ or t-) -> what they add
            auto each = [&](auto share) {
#pragma unroll
                for (int j = 0; j < NI; ++j) {
                    const int o = (int)b0 + (wc * NI + j) * 32 + fl, oc = o < O ? o : O - 1;
                    float sp = 0.0f, sn = 0.0f;
#pragma unroll
                    for (int i = 0; i < MI; ++i) {
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            const int k = (block_of(i, q) >> sh) * 2 + fh, jb = block_of(i, q) & (per - 1);
                            const float2 tt = g.tT[(int64_t)(k < K ? k : K - 1) * Op + oc];
                            const float4 r = make_float4(acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2],
                                                         acc[i][j][4 * q + 3]);
                            sp += share(jb, r, tt.x);
                            sn += share(jb, r, tt.y);
                            if (jb == per - 1) {
                                store(k, o, sp, sn);
                                sp = sn = 0.0f;
                            }
                            if (q & 1) fence();
                        }
                    }
                }
            };
            if (harm) {
                each([&](int jb, float4 r, float tv) {
                    const float th = ((float)h.wc + (float)h.wh * tv) * (h.lut_scale * (float)(jb + 1));
                    const float f = th - floorf(th);
                    const float2 u = sep_kink_functions(h, tv);
                    return __builtin_amdgcn_cosf(f) * fmaf(r.y, u.y, r.x * u.x) +
                           __builtin_amdgcn_sinf(f) * fmaf(r.w, u.y, r.z * u.x);
                });
            } else {
                each([&](int jb, float4 r, float tv) {
                    const float2 u = sep_cheb_from(first + 4 * jb, tv);
                    const float u2 = fmaf(2.0f * tv, u.y, -u.x), u3 = fmaf(2.0f * tv, u2, -u.y);
                    return fmaf(r.w, u3, fmaf(r.z, u2, fmaf(r.y, u.y, r.x * u.x)));
                });
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
// the launches that return, 7 to 12 us (tables 1 to 5: their assignment passes are one launch) where the
// sample refuses it (sep_sample_refuses), and the statistics, 10 to 20 us, where only they do (one threshold
// or input far from the others). The lines lie where the first is 1% of the call; the second is then 2% of
// it for the formula and up to 5% for tables. Measured (us, forward / backward, without the contraction
// against refused): formula, 192 x 768 at 2^29 cells over 4 V 526 / 976 against 532 / 985, one outlier
// 525 / 977 against 537 / 993; tables, 384 x 1536 at 2^30 over 5 V 376 / 801 against 380 / 803, one
// outlier 347 / 738 against 366 / 761, 768 x 3072 at 4096 tokens 2256 / 5115 against 2278 / 5125. Taken
// calls gain from far smaller sizes on: formula, 192 x 768 at 2^25.2 65 / 101 against 45 / 78, at 2^27.2
// 157 / 288 against 52 / 106 (refused there 163 / 296).
#ifndef ISA_EKV_CONTRACT_MIN_CELLS
#define ISA_EKV_CONTRACT_MIN_CELLS (1 << 29)
#endif
// Table calls (us, forward / backward, per-cell kernels against the contraction), 384 x 1536: at 2^30
// cells 333 / 565 against 177 / 458 (4096 entries) and 339 / 606 against 160 / 414 (8192) at the initial
// thresholds, over 1 V (16 terms) 343 against 242 (4096, forward) and 352 / 716 against 221 / 570 (8192);
// at 2^29 222 / 331 against 122 / 271, and 227 / 408 against 234 / 409 over 5 V (refused).
#ifndef ISA_EKV_CONTRACT_MIN_CELLS_LUT
#define ISA_EKV_CONTRACT_MIN_CELLS_LUT (1 << 30)
#endif

struct SepPlan {
    int max_terms;  // 0: not considered
    bool big;       // 256 x 256 tiles instead of 128 x 128
    int split;                     // forward
    int split_dx[4], split_dv[4];  // backward: of the harmonics, the singles, pairs and triples
    int planes_dx, planes_dv;
    int64_t Kp, Op;
    size_t off_head, off_part, off_tab, off_tab2, off_tabE, off_lut, off_xop, off_wop, off_xcls[4], off_wcls[4], off_gop,
        off_gops, off_gopT, off_gopTs, off_tT, off_planes, off_planes_dv, bytes;
};

constexpr int64_t kSepOperandBytes = ((int64_t)4 << 30) - (1 << 20);  // of one operand, at most (32-bit byte offsets)
// Of a call's operands and planes, at most (3% of the card). With 4096 entries a GPT-L layer's 768 -> 3072
// stays below both limits up to 87300 tokens forward and 69800 backward, 3072 -> 768 up to 21800 and 29500;
// larger calls run the per-cell kernels.
constexpr size_t kSepPlanBytes = (size_t)8 << 30;

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

// The plan for up to `terms` terms; max_terms 0 where an operand would be too large.
SepPlan plan_sep_terms(int lut_n, int64_t M, int64_t K, int64_t O, bool backward, bool need_x, bool need_w, size_t base,
                       int terms) {
    SepPlan p{};
    p.bytes = base;
    p.Kp = round_up(K, 8);
    p.Op = round_up(O, 256);
    const int64_t Mi = sep_inner(M), Oi = sep_inner(O), Kr = sep_inputs(K);
    const bool lut = lut_n > 0;
    const int most = lut ? kSepMaxHarmonics : 0;  // the device takes as many harmonics as the table needs
    // (a backward's widest operand: dVth's triples, six bytes a value, or the harmonics; or G's triples)
    const int64_t widest = backward ? std::max(std::max(Mi, Oi) * Kr * std::max(6 * sep_classes(terms, true).n3, 8 * most),
                                               Mi * Oi * 6)
                                    : std::max(M, O) * SepRow(K, terms, most).bytes;
    if (widest >= kSepOperandBytes) return p;
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
    if (lut) {
        p.off_lut = take((int64_t)lut_n * 16 + 256 * 16);
        p.off_tabE = take((int64_t)kSepGridMax * 8);
    }
    if (!backward) {
        const int64_t row = std::max(SepRow(K, terms, most).bytes, SepRow(K, 8, most).bytes);
        p.off_xop = take(M * row);
        p.off_wop = take(O * row);
        const int64_t slabs = SepRow(K, 8, most).bytes / 112;
        p.big = sep_big(M, O, slabs);
        const int64_t tile = p.big ? 256 : 128;
        p.split = sep_splits(((M + tile - 1) / tile) * ((O + tile - 1) / tile), slabs, p.big, 8.0 * M * O);
        p.off_planes = take((int64_t)p.split * M * O * 4);
    } else {
        p.off_tab2 = take((int64_t)kSepGridMax * 4 * terms);
        if (need_x) {
            p.off_gop = take(M * Oi * 6);
            p.off_gops = take(M * Oi * 2);
        }
        if (need_w) {
            p.off_gopT = take(O * Mi * 6);
            p.off_gopTs = take(O * Mi * 2);
        }
        auto values = [&](int c, bool dv, int r) { return c == 0 ? 4 * most : sep_classes(r, dv).count(c); };
        auto slabs = [&](int c, int64_t inner) { return inner / (c == 0 ? 64 : c == 3 ? 16 : 64 / c); };
        auto tiles = [&](int c, bool dv, int64_t tile) {  // at 8 terms
            return (sep_rows(K, values(c, dv, 8)) + tile - 1) / tile * (((dv ? O : M) + tile - 1) / tile);
        };
        // the work of both gradients in slabs of 256 x 256 tiles: 64 per CU take them (16384 tokens, 384 x
        // 1536, 4096 entries: 1.93 ms against 2.16 with 128 x 128), whichever gradient the call wants, so
        // that each has the same bits
        int64_t work = 0;
        for (int c = 0; c < 4; ++c) work += tiles(c, false, 256) * slabs(c, Oi) + tiles(c, true, 256) * slabs(c, Mi);
        p.big = work >= 64 * kCUs && K >= 64 && M >= 192 && O >= 192;
        for (int c = 0; c < 4; ++c) {  // the harmonics, singles, pairs, triples
            const int bytes = c == 0 ? 2 : 2 * c;
            const int vx = std::max(values(c, false, 8), values(c, false, terms));
            const int vw = std::max(values(c, true, 8), values(c, true, terms));
            if (vx == 0) continue;
            if (need_w) p.off_xcls[c] = take(Kr * vw * Mi * bytes);
            if (need_x) p.off_wcls[c] = take(Kr * vx * Oi * bytes);
            const int64_t tile = p.big ? 256 : 128;
            p.split_dx[c] = sep_splits(tiles(c, false, tile), slabs(c, Oi), p.big, 8.0 * M * K);
            p.split_dv[c] = sep_splits(tiles(c, true, tile), slabs(c, Mi), p.big, 16.0 * p.Kp * p.Op);
            p.planes_dx += p.split_dx[c];
            p.planes_dv += p.split_dv[c];
        }
        p.off_tT = take(K * p.Op * 8);
        if (need_x) p.off_planes = take((int64_t)p.planes_dx * M * K * 4);
        if (need_w) p.off_planes_dv = take((int64_t)p.planes_dv * 2 * p.Kp * p.Op * 4);
    }
    p.bytes = off;
    return p;
}

// lut_n: table entries, 0 for the formula.
SepPlan plan_sep(int lut_n, int64_t M, int64_t K, int64_t O, bool backward, bool need_x, bool need_w, size_t base) {
    SepPlan none{};
    none.bytes = base;
    const double cells = (double)M * (double)K * (double)O;
    if (M < 16 || O < 16 || K < 8 || (backward && !need_x && !need_w) ||
        cells < (double)(lut_n > 0 ? (int64_t)ISA_EKV_CONTRACT_MIN_CELLS_LUT : (int64_t)ISA_EKV_CONTRACT_MIN_CELLS) ||
        (lut_n > 0 && (lut_n < kSepLutMin || lut_n > kSepLutMax)))
        return none;
    for (int terms = backward && lut_n > 0 && lut_n < kSepLutWideMin ? 8 : kSepMaxTerms; terms >= 8; terms /= 2) {
        const SepPlan p = plan_sep_terms(lut_n, M, K, O, backward, need_x, need_w, base, terms);
        if (p.max_terms > 0 && p.bytes - base < kSepPlanBytes) return p;
    }
    return none;
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
    a.lut_info = reinterpret_cast<float4*>(ws + p.off_lut);
    a.lut_val = reinterpret_cast<double2*>(ws + p.off_lut + 256 * 16);
    a.max_terms = p.max_terms;
}

void sep_point_forward(const SepPlan& p, SepArgs& a, char* ws) {
    sep_point(p, a, ws);
    a.xop = ws + p.off_xop;
    a.wop = ws + p.off_wop;
}

// The forward's operands (and, where it does not take the call, the per-cell kernels' prep).
hipError_t sep_forward_operands(const SepPlan& p, SepArgs a, const PrepArgs& prep, char* ws, hipStream_t s) {
    sep_point_forward(p, a, ws);
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
    sep_point_forward(p, a, ws);
    SepGemm g{};
    g.head = a.head;
    g.M = a.M;
    g.K = a.K;
    g.O = a.O;
    g.n = 1;
    g.p[0] = SepProduct{a.xop, a.wop, kSepForward, 0, a.M, a.O, 0, p.split, reinterpret_cast<float*>(ws + p.off_planes)};
    const int64_t tile = p.big ? 256 : 128;
    launch_sep_gemm<true>(p.big, (unsigned)((a.M + tile - 1) / tile * ((a.O + tile - 1) / tile) * p.split), g, s);
    return hipGetLastError();
}

void sep_point_backward(const SepPlan& p, SepArgs& a, char* ws) {
    sep_point(p, a, ws);
    a.tab2 = reinterpret_cast<float*>(ws + p.off_tab2);
    // (harmonics last)
    for (int c = 0; c < 4; ++c) {
        a.xcls[(c + 3) % 4] = ws + p.off_xcls[c];
        a.wcls[(c + 3) % 4] = ws + p.off_wcls[c];
    }
    a.gop = ws + p.off_gop;
    a.gops = ws + p.off_gops;
    a.gopT = ws + p.off_gopT;
    a.gopTs = ws + p.off_gopTs;
    a.tT = reinterpret_cast<float2*>(ws + p.off_tT);
    a.Op = p.Op;
}

// The backward's operands; glue: the layer glue's gradient pass, which writes a.g.
hipError_t sep_backward_operands(const SepPlan& p, SepArgs a, const PrepArgs& prep, const GlueGradArgs* glue, char* ws,
                                 hipStream_t s) {
    sep_point_backward(p, a, ws);
    const int64_t stat = kSepStatX + kSepStatW + (a.lut_n + 255) / 256 + (glue ? (int64_t)kGlueBlocks * (glue->Op / 256) : 0);
    hipLaunchKernelGGL(sep_stat_kernel, dim3((unsigned)stat), dim3(256), 0, s, a, prep,
                       glue ? *glue : GlueGradArgs{});
    hipLaunchKernelGGL(sep_table_kernel, dim3((unsigned)(kSepTableBlocks + kSepStatG)), dim3(256), 0, s, a);
    const int64_t kt = (a.K + 31) / 32, ot = (a.O + 127) / 128;
    const int64_t x_blocks = a.need_w ? kt * ((a.M + 127) / 128) : 0, w_blocks = kt * ot, g_blocks = ot * (sep_inner(a.M) / 32);
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
    g.x = a.x;
    g.in_affine = a.in_affine;
    g.in_lo = a.in_lo;
    g.in_hi = a.in_hi;
    g.tab2 = a.tab2;
    g.tabE = a.tabE;
    g.tT = a.tT;
    const int64_t tile = p.big ? 256 : 128;
    int64_t blocks = 0;
    auto add = [&](int kind, int parts, const char* x, const char* y, int64_t b_rows, int64_t inner, int split, float*& out,
                   int64_t plane) {
        g.p[g.n++] = SepProduct{x, y, kind, parts, a.K, b_rows, inner, split, out};
        out += split * plane;
        int64_t rows = 0;  // at the most that the device may choose
        for (int r = 8; r <= p.max_terms; r *= 2) rows = std::max(rows, sep_rows(a.K, sep_values(kind, parts, r, kSepMaxHarmonics)));
        blocks += (rows + tile - 1) / tile * ((b_rows + tile - 1) / tile) * split;
    };
    float* dx = reinterpret_cast<float*>(ws + p.off_planes);
    float* dv = reinterpret_cast<float*>(ws + p.off_planes_dv);
    const int64_t px = a.M * a.K, pv = 2 * p.Kp * p.Op;
    for (const int c : {3, 2, 1, 0}) {  // the longest first; the harmonics' planes are the last ones
        if (p.split_dx[c] == 0) continue;
        const int at = (c + 3) % 4;
        if (a.need_x) add(kSepDx, c, a.wcls[at], c >= 2 ? a.gop : a.gops, a.M, sep_inner(a.O), p.split_dx[c], dx, px);
        if (a.need_w) add(kSepDv, c, a.xcls[at], c >= 2 ? a.gopT : a.gopTs, a.O, sep_inner(a.M), p.split_dv[c], dv, pv);
    }
    launch_sep_gemm<false>(p.big, (unsigned)blocks, g, s);
    return hipGetLastError();
}
