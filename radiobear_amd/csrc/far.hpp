// Forward line sums with far-line series, FP32 and FP64 modes (included by alpha.hip, after
// the line-sum kernel it replaces when the series are on).
//
// A line's term is a rational function of x = f^2 with two poles p (the roots of its
// denominator x^2 - 2 Ds x + P0, P0 = Ds^2 + h):
//   term(x) = (a x + c) / (x^2 - 2 Ds x + P0).
// Over a wavefront tile whose columns span x in [lo, hi]:
//   * every |p| <= kFarRatio lo ("below"): term = sum_k m_k x^-(k+1), with
//     m_0 = a, m_1 = c + 2 Ds a, m_k = 2 Ds m_{k-1} - P0 m_{k-2};
//   * every |p| >= hi / kFarRatio ("above"): term = sum_k n_k x^k, with
//     n_0 = c / P0, n_1 = (a + 2 Ds n_0) / P0, n_k = (2 Ds n_{k-1} - n_{k-2}) / P0
// (the recurrences match powers of x in term * denominator = a x + c).  kFarTerms = 16
// terms at kFarRatio = 1/3 leave ~4e-8 of a far line's value for two well-separated
// poles and at most 8e-7 at the ratio limit for a near-double pole of a Gross line
// (a = 0: 15 terms carry it, with coefficients growing like (k + 1) p^k); far lines are
// small next to the near ones, and the tables stay within 3e-7 of FP64 like the direct
// FP32 sums.  On 800 layers x 1024 frequencies (0.3-300 GHz, 128-column tiles) about
// 30 % of the (line, tile) pairs are neither: only those go to the near pass.  (12
// terms at 1/4 leave more near pairs, 33 %, and were 2 % slower overall.)  FP64 mode uses
// the same 16 terms at ratio 0.15 (at most ~8e-12 of a far line's value) and sums its near
// lines in FP64 from their (D, a, c, g, G).
//
// alpha_prep_kernel (one thread per layer and deriver) first writes every layer's
// coefficient derivers to the workspace; both passes below read them from there.
// alpha_far_kernel (block = layer x group of kFarTiles tiles x part of the layer's
// staging rounds; each wavefront a contiguous run of 64-line blocks): each lane derives
// one line's coefficients per coefficient set (once per line and layer, its catalogue
// columns fetched a block ahead), classifies it against every tile of the group (one
// ballot per tile gives the tiles' near-mask words) and adds its series to running sums
// keyed by the first tile it is below for and the last it is above for (prefix and
// suffix sums over the tiles give each tile's moments).  The h2o base term is summed
// here.
// alpha_near_kernel (block = tile x layer, all four wavefronts on the tile's
// columns): lists the tile's near lines from its masks, derives each listed line's
// coefficients again from its catalogue row (the catalogue stays in L2; no per-layer copy
// of the lines goes through HBM), sums them at the nodes of column intervals they are well
// away from and at the columns they are close to, with the lines split between the
// wavefronts, adds the wavefronts in order and the series of the summed moments, and
// writes the same per-slot partials the finish kernel reads (one part).

constexpr int kFarTerms = 16;
// pole ratio of a far line: 1/3 in FP32 mode, 0.15 in FP64 mode (at most ~8e-12 of a far
// line's value there, against the 1e-9 FP64 parity bar)
template <bool F32>
__host__ __device__ constexpr double far_ratio() { return F32 ? 1.0 / 3.0 : 0.15; }
constexpr int kFarTiles = 8;                          // tiles per alpha_far_kernel block
constexpr int kFarSets = 6;                           // h2o, h2s, inversion set 0, set 1, rot + v2, ph3
constexpr int kFarMom = kFarSets * 2 * kFarTerms;     // moments per (layer, part, tile)
constexpr int kSegStream[kSegs] = {0, 1, 2, 4, 5, 6};
constexpr int kSegFarSet[kSegs] = {0, 1, 2, 4, 4, 5};
constexpr int kSegVar[kSegs] = {0, 0, 1, 1, 1, 0};    // columns' x (0) or x for NH3 (1)
constexpr int kListWords = 112;                       // mask words listed per window (near_sum; with 128 the
                                                      // widest FP32 tile's block is past a quarter of a CU's LDS)
constexpr int kFarRanges = 4;                         // x; x NH3; x NH3 of set 0 columns; of set 1

__device__ inline void tile_cols(const AlphaArgs &A, int tile, int &c0, int &c1) {
    c0 = tile * A.tile_width;
    c1 = min(c0 + A.tile_width, A.nf);
}

// inversion coefficient sets a tile's columns use: bit 0 set 0 (columns < nf_low), bit 1 set 1
__device__ inline int tile_sets(const AlphaArgs &A, int c0, int c1) {
    return (c0 < min(c1, A.nf_low) ? 1 : 0) | (max(c0, A.nf_low) < c1 ? 2 : 0);
}

// [lo, hi] of x, x for NH3, and x for NH3 over the set 0 / set 1 columns of a tile
// (called by a whole wavefront; the results are wavefront-uniform, +inf/-inf when empty)
__device__ inline void tile_ranges(const AlphaArgs &A, int tile, double (&lo)[kFarRanges],
                                   double (&hi)[kFarRanges]) {
#pragma unroll
    for (int v = 0; v < kFarRanges; ++v) {
        lo[v] = INFINITY;
        hi[v] = -INFINITY;
    }
    int c0, c1;
    tile_cols(A, tile, c0, c1);
    for (int c = c0 + static_cast<int>(threadIdx.x % 64); c < c1; c += 64) {
        const double f = A.freq[c];
        const double fn = A.freq_nh3 ? A.freq_nh3[c] : f;
        const double xs[kFarRanges] = {f * f, fn * fn, c < A.nf_low ? fn * fn : NAN, c < A.nf_low ? NAN : fn * fn};
#pragma unroll
        for (int v = 0; v < kFarRanges; ++v) {
            lo[v] = fmin(lo[v], xs[v]);   // fmin / fmax skip the NaN placeholders
            hi[v] = fmax(hi[v], xs[v]);
        }
    }
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) {
#pragma unroll
        for (int v = 0; v < kFarRanges; ++v) {
            lo[v] = fmin(lo[v], __shfl_xor(lo[v], m));
            hi[v] = fmax(hi[v], __shfl_xor(hi[v], m));
        }
    }
}

// moduli (smaller rs, larger rb) of the two roots of x^2 - 2 Ds x + P0, P0 = Ds^2 + h:
// a complex pair of modulus sqrt(P0) when h >= 0, else |Ds| -+ sqrt(-h); in FP32 from the
// FP64 coefficients (the class tests compare FP32 values; NaN coefficients give NaN
// moduli, near everywhere)
__device__ inline void pole_moduli_f32(double Ds, double h, double P0, float &rs, float &rb) {
    const float m = fabsf(static_cast<float>(Ds)), q = __builtin_amdgcn_sqrtf(fabsf(static_cast<float>(h)));
    const float r = __builtin_amdgcn_sqrtf(static_cast<float>(P0));
    const bool complex_pair = h >= 0.0;
    rb = complex_pair ? r : m + q;
    rs = complex_pair ? r : fabsf(m - q);
    if (!(h == h)) rs = rb = NAN;
}

// a copy of a wavefront-uniform value held in scalar registers (each 32-bit word taken from
// the first active lane)
template <class T>
__device__ __forceinline__ T uniform(const T &v) {
    static_assert(sizeof(T) % 4 == 0, "whole 32-bit words");
    T out = v;
    const int *src = reinterpret_cast<const int *>(&v);
    int *dst = reinterpret_cast<int *>(&out);
#pragma unroll
    for (int w = 0; w < static_cast<int>(sizeof(T) / 4); ++w) dst[w] = __builtin_amdgcn_readfirstlane(src[w]);
    return out;
}

// b when second, else a, chosen word by word: choosing between the two objects' addresses
// instead makes the compiler keep both in scratch and read the chosen one from there
template <class T>
__device__ __forceinline__ T pick(const T &a, const T &b, bool second) {
    static_assert(sizeof(T) % 4 == 0, "whole 32-bit words");
    T out = a;
    const int *wa = reinterpret_cast<const int *>(&a), *wb = reinterpret_cast<const int *>(&b);
    int *wo = reinterpret_cast<int *>(&out);
#pragma unroll
    for (int w = 0; w < static_cast<int>(sizeof(T) / 4); ++w) wo[w] = second ? wb[w] : wa[w];
    return out;
}

// The segments' coefficient derivers per layer (the layer's powers of T and partial pressures,
// computed once by alpha_prep_kernel): [nl][kSegs][kPrepWords] doubles, set 0's deriver in
// words 0-7, set 1's (the same one outside the nh3_hs inversion lines) in 8-15, and their FP32
// weight scales (1 in FP64 mode) in 16 and 17.  The passes read a layer's row with uniform loads.
constexpr int kPrepWords = 18;
template <int S>
using SegC = std::integral_constant<int, S>;

// One thread per (deriver, layer), derivers slowest: the lanes of a wavefront build the same
// deriver (with the layer slowest they ran all six one after the other), and the nh3_hs inversion
// lines' two sets are two derivers.  A wavefront per block spreads the few of them over the CUs.
// The powers' latency bounds it: 800 layers 20 -> 9 us, 400 layers 22 -> 9 us.
constexpr int kPrepThreads = 64;
constexpr int kPrepDerivers = kSegs + 1;   // kSegs: the inversion lines' set 1

template <bool F32>
__global__ __launch_bounds__(kPrepThreads) void alpha_prep_kernel(AlphaArgs A) {
    const long long e = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (e >= static_cast<long long>(A.nl) * kPrepDerivers) return;
    const int layer = static_cast<int>(e % A.nl), which = static_cast<int>(e / A.nl);
    const int seg = which == kSegs ? 2 : which;
    const LayerT<double> L = layer_of(A, layer);
    const DevBlock *blk = A.cat.blk;
    double *row = A.far_prep + (static_cast<size_t>(layer) * kSegs + seg) * kPrepWords;
    // the deriver into set s's words, its weight scale into word 16 + s
    auto put = [&](int s, const auto &p, double sc) {
        using Prep = std::decay_t<decltype(p)>;
        static_assert(sizeof(Prep) <= 8 * sizeof(double) && sizeof(Prep) % sizeof(double) == 0,
                      "a deriver is at most 8 doubles");
        const double *w = reinterpret_cast<const double *>(&p);
        for (int k = 0; k < 8; ++k) row[8 * s + k] = k < static_cast<int>(sizeof(Prep) / sizeof(double)) ? w[k] : 0.0;
        row[16 + s] = F32 ? sc : 1.0;
    };
    auto one = [&](const auto &p, int kind) {   // segments of one set: both halves the same
        put(0, p, pow2_scale(p.pref * blk[kind].wscale));
        put(1, p, 1.0);
    };
    switch (which) {
        case 0: one(H2oPrep<double>(L), RBX_LINES_H2O); break;
        case 1: one(H2sPrep<double>(L), RBX_LINES_H2S); break;
        case 2:
        case kSegs: {
            const int s = which == kSegs ? 1 : 0;
            const InvPrep<double> p(L, s ? 1 : nh3_low_set(A.abs.nh3));
            put(s, p, pow2_scale(p.pref * blk[RBX_LINES_NH3_INV].wscale));
            break;
        }
        case 3: one(RotPrep<double>(L), RBX_LINES_NH3_ROT); break;
        case 4: one(V2Prep<double>(L), RBX_LINES_NH3_V2); break;
        default: one(Ph3Prep<double>(L), RBX_LINES_PH3); break;
    }
}

// a deriver from its table words (in scalar registers)
template <class Prep>
__device__ __forceinline__ Prep load_prep(const double *w) {
    struct Raw {
        double v[sizeof(Prep) / sizeof(double)];
    } r;
#pragma unroll
    for (int k = 0; k < static_cast<int>(sizeof(Prep) / sizeof(double)); ++k) r.v[k] = w[k];
    return uniform(__builtin_bit_cast(Prep, r));
}

// f(segment as a compile-time constant, set 0 deriver, set 1 deriver, scale 0, scale 1) with
// the layer's derivers of the segment from the table
template <class F>
__device__ __forceinline__ void with_prep(const AlphaArgs &A, int layer, int seg, F &&f) {
    const double *row = A.far_prep + (static_cast<size_t>(layer) * kSegs + seg) * kPrepWords;
    const double s0 = __builtin_amdgcn_readfirstlane(row[16]), s1 = __builtin_amdgcn_readfirstlane(row[17]);
    switch (seg) {
        case 0: {
            const auto p = load_prep<H2oPrep<double>>(row);
            f(SegC<0>{}, p, p, s0, s1);
            break;
        }
        case 1: {
            const auto p = load_prep<H2sPrep<double>>(row);
            f(SegC<1>{}, p, p, s0, s1);
            break;
        }
        case 2: {
            const auto p0 = load_prep<InvPrep<double>>(row), p1 = load_prep<InvPrep<double>>(row + 8);
            f(SegC<2>{}, p0, p1, s0, s1);
            break;
        }
        case 3: {
            const auto p = load_prep<RotPrep<double>>(row);
            f(SegC<3>{}, p, p, s0, s1);
            break;
        }
        case 4: {
            const auto p = load_prep<V2Prep<double>>(row);
            f(SegC<4>{}, p, p, s0, s1);
            break;
        }
        default: {
            const auto p = load_prep<Ph3Prep<double>>(row);
            f(SegC<5>{}, p, p, s0, s1);
            break;
        }
    }
}

// coefficient set v of line i of a segment from its catalogue row (both passes derive a
// line's coefficients this way; `base` collects the h2o base term)
template <class Prep, class Row>
__device__ __forceinline__ CoefT<double> seg_coef(const Prep &p0, const Prep &p1, int v, const Row &row, int i,
                                                  double &base) {
    if constexpr (Prep::kShared) {
        const double w = p0.weight(row, i);
        return v ? p1.coef(row, i, w) : p0.coef(row, i, w);
    } else {
        return p0(row, i, base);
    }
}

// ---- pass 1: far-line series and near masks ----
//
// A line's series coefficients (m_k below, n_k above) do not depend on the tile, only its
// class does: the line is below for the tiles with q lo >= its larger pole modulus and
// above for those with hi / q <= its smaller one.  Ranked by q lo, the tiles a line is
// below for are the last ones (all ranks >= kb, kb = the number of tiles with q lo under
// the modulus); ranked by hi / q, the tiles it is above for are the first ka.  So each
// thread derives its own line's series once per coefficient set and adds them into a
// difference array over the ranks (entry kb of the below array, entry ka of the above
// one); the moments of a tile are the prefix (below) or suffix (above) sums at its rank.
// The line lists are sorted by centre, so a thread's successive lines mostly share kb
// and ka: it keeps running sums in registers for its current kb and ka and adds them to
// the block's difference arrays in LDS (FP64 atomics) only when they change.  Near bits
// come from one wavefront ballot per tile.

constexpr int kFarWaves = kThreads / 64;

struct FarShared {
    // per wavefront: difference arrays, below (entry kb) and above (entry ka)
    double dB[kFarWaves][kFarTiles + 1][kFarTerms];
    double dA[kFarWaves][kFarTiles + 1][kFarTerms];
    double mom[kFarTiles][kFarMom];
    double lo[kFarTiles][kFarRanges], hi[kFarTiles][kFarRanges];
    double bsum[kThreads / 64];
    alignas(16) float thr[2][kFarTiles];   // current coefficient set: q lo, hi / q (+inf: unused)
};

// a used tile's class thresholds for range rv: q lo (below) and hi / q (above), as FP32
template <bool F32>
__device__ inline float far_threshold(const FarShared &sh, int j, int rv, bool above) {
    const double q = far_ratio<F32>();
    return above ? static_cast<float>(sh.hi[j][rv] / q) : static_cast<float>(q * sh.lo[j][rv]);
}

// rank of used tile j among the used tiles by its threshold (ties by index)
template <bool F32>
__device__ inline int tile_rank(const FarShared &sh, unsigned used, int j, int rv, bool above) {
    const float vj = far_threshold<F32>(sh, j, rv, above);
    int r = 0;
#pragma unroll
    for (int i = 0; i < kFarTiles; ++i) {
        const float vi = far_threshold<F32>(sh, i, rv, above);
        r += ((used >> i) & 1u) && (vi < vj || (vi == vj && i < j)) ? 1 : 0;
    }
    return r;
}


// The lanes with `pred` add their running sums acc into entry e (their own) of the
// wavefront's difference array d: for each entry among them, the 16 terms are summed over
// its lanes by a fixed reduce-scatter (halving the terms each lane carries at xor 32, 16, 8
// and 4, then adding over xor 2 and 1: term 8 b5 + 4 b4 + 2 b3 + b2 ends in the lanes with
// those lane bits), so the result does not depend on timing.  Called by the whole wavefront.
__device__ __forceinline__ void far_flush(double (&d)[kFarTiles + 1][kFarTerms], bool pred, int e,
                                          const double (&acc)[kFarTerms]) {
    static_assert(kFarTerms == 16, "the reduce-scatter below is written for 16 terms");
    unsigned long long rem = __ballot(pred);
    const int lane = threadIdx.x % 64;
    const bool b5 = lane & 32, b4 = lane & 16, b3 = lane & 8, b2 = lane & 4;
    while (rem != 0ull) {
        const int b = __builtin_amdgcn_readlane(e, __builtin_ctzll(rem));
        const bool sel = pred && e == b;
        rem &= ~__ballot(sel);
        double w8[8], w4[4], w2[2];
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const double lo = sel ? acc[t] : 0.0, hi = sel ? acc[t + 8] : 0.0;
            w8[t] = (b5 ? hi : lo) + __shfl_xor(b5 ? lo : hi, 32);
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) w4[t] = (b4 ? w8[t + 4] : w8[t]) + __shfl_xor(b4 ? w8[t] : w8[t + 4], 16);
#pragma unroll
        for (int t = 0; t < 2; ++t) w2[t] = (b3 ? w4[t + 2] : w4[t]) + __shfl_xor(b3 ? w4[t] : w4[t + 2], 8);
        double w1 = (b2 ? w2[1] : w2[0]) + __shfl_xor(b2 ? w2[0] : w2[1], 4);
        w1 += __shfl_xor(w1, 2);
        w1 += __shfl_xor(w1, 1);
        if ((lane & 3) == 0) d[b][(b5 ? 8 : 0) + (b4 ? 4 : 0) + (b3 ? 2 : 0) + (b2 ? 1 : 0)] += w1;
    }
}

template <bool F32>
__global__ __launch_bounds__(kThreads, 3) void alpha_far_kernel(AlphaArgs args) {
    // the arguments read where the launch put them (explicit kernel arguments open the
    // kernarg segment): a private copy of the struct would be spilled to scratch per lane
#if defined(__HIP_DEVICE_COMPILE__)
    const AlphaArgs &A = *reinterpret_cast<const AlphaArgs *>(__builtin_amdgcn_kernarg_segment_ptr());
#else
    const AlphaArgs &A = args;   // (host pass: never run)
#endif
    __shared__ FarShared sh;
    const int ngroups = (A.tiles_total + kFarTiles - 1) / kFarTiles;
    const int layer = blockIdx.x / ngroups, g = blockIdx.x % ngroups;
    const int part = blockIdx.y, nsplit = gridDim.y;
    const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
    const LayerT<double> L = layer_of(A, layer);

    for (int j = wave; j < kFarTiles; j += kThreads / 64) {
        double lo[kFarRanges], hi[kFarRanges];
        tile_ranges(A, g * kFarTiles + j, lo, hi);   // empty for tiles past the last
        if (lane == 0) {
#pragma unroll
            for (int v = 0; v < kFarRanges; ++v) {
                sh.lo[j][v] = lo[v];
                sh.hi[j][v] = hi[v];
            }
        }
    }
    for (int e = tid; e < kFarTiles * kFarMom; e += kThreads) (&sh.mom[0][0])[e] = 0.0;
    for (int e = tid; e < kFarWaves * (kFarTiles + 1) * kFarTerms; e += kThreads) {
        (&sh.dB[0][0][0])[e] = 0.0;
        (&sh.dA[0][0][0])[e] = 0.0;
    }
    int gc0, gc1;
    tile_cols(A, g * kFarTiles, gc0, gc1);
    gc1 = min(A.nf, (g + 1) * kFarTiles * A.tile_width);
    const int gsets = tile_sets(A, gc0, gc1);   // inversion sets any tile of the group needs
    const int ntiles = min(kFarTiles, A.tiles_total - g * kFarTiles);
    unsigned tile_set_bits[2] = {0u, 0u};       // tiles of the group whose columns use set 0 / 1
    for (int jj = 0; jj < ntiles; ++jj) {
        int c0, c1;
        tile_cols(A, g * kFarTiles + jj, c0, c1);
        const int ts = tile_sets(A, c0, c1);
        tile_set_bits[0] |= (ts & 1) ? 1u << jj : 0u;
        tile_set_bits[1] |= (ts & 2) ? 1u << jj : 0u;
    }
    __syncthreads();

    const LinePlan plan(A, L.P);
    const int r0 = plan.begin(part, nsplit), r1 = plan.begin(part + 1, nsplit);
    double base = 0.0;
    int off = 0;
#pragma unroll 1
    for (int seg = 0; seg < kSegs; ++seg) {
        const int a0 = max(r0, off), b0 = min(r1, off + plan.nr[seg]);
        const int seg_off = off;
        off += plan.nr[seg];
        if (a0 >= b0) continue;
        with_prep(A, layer, seg, [&](auto segc, const auto &p0, const auto &p1, double s0, double s1) {
            constexpr int SEG = decltype(segc)::value;
            constexpr bool inv = SEG == 2;
            const DevBlock &B = A.cat.blk[kSegKind[SEG]];
            const int need = inv ? gsets : 1;
            (void)s0;
            (void)s1;
#pragma unroll 1
            for (int v = 0; v < 2; ++v) {
                if (!((need >> v) & 1)) continue;
                const unsigned used = inv ? tile_set_bits[v] : (1u << ntiles) - 1u;
                const int nv = __popc(used);
                const int rv = kSegVar[SEG] == 0 ? 0 : (inv ? 2 + v : 1);
                // thresholds of the used tiles; unused ones never count (+inf: a finite
                // modulus is below it and never at or above it)
                if (tid < 2 * kFarTiles) {
                    const int j = tid % kFarTiles;
                    sh.thr[tid / kFarTiles][j] = (used >> j) & 1u ? far_threshold<F32>(sh, j, rv, tid >= kFarTiles) : INFINITY;
                }
                __syncthreads();
                const int soff = A.far_off[kSegStream[SEG] + ((inv && v) ? 1 : 0)];
                unsigned int *mrow = A.near + (static_cast<size_t>(layer) * A.tiles_total + g * kFarTiles) * A.far_words + soff;
                double accB[kFarTerms], accA[kFarTerms];
#pragma unroll
                for (int k = 0; k < kFarTerms; ++k) accB[k] = accA[k] = 0.0;
                int cbB = -1, cbA = -1;   // entries the running sums belong to (-1: none yet)
                // wavefront w takes a contiguous run of the part's 64-line blocks (its lanes'
                // successive lines are 64 apart, so their entries change seldom)
                const int nblk = b0 - a0;   // blocks per wavefront (kThreads / 64 per round)
                const int blk0 = (a0 - seg_off) * kFarWaves + wave * nblk;
                // the set-v deriver, chosen once for the part's lines
                const auto pv = pick(p0, p1, v != 0);
                // each line's catalogue columns are fetched one block ahead
                LineRow<kNumCols[kSegKind[SEG]]> next;
                next.load(B, min(blk0 * 64 + lane, B.n - 1));
#pragma unroll 1
                for (int blk = blk0; blk < blk0 + nblk; ++blk) {
                    const int i = blk * 64 + lane;
                    const bool valid = i < B.n;
                    const auto row = next;
                    if (blk + 1 < blk0 + nblk) next.load(B, min(i + 64, B.n - 1));
                    CoefT<double> c = {0.0, 0.0, 0.0, 0.0, 1.0};
                    if (valid) c = seg_coef(p0, pv, 1, row, i, base);
                    double Ds, h;
                    shifted_denominator(c, Ds, h);
                    const double P0 = fma(Ds, Ds, h);
                    // class against every used tile: below when rb <= q lo, else above when
                    // rs >= hi / q, else near (NaN moduli: near everywhere)
                    float frs, frb;
                    pole_moduli_f32(Ds, h, P0, frs, frb);
                    float loq[kFarTiles], hiq[kFarTiles];
#pragma unroll
                    for (int j = 0; j < kFarTiles; j += 4) {
                        const float4 l4 = *reinterpret_cast<const float4 *>(&sh.thr[0][j]);
                        const float4 h4 = *reinterpret_cast<const float4 *>(&sh.thr[1][j]);
                        loq[j] = l4.x; loq[j + 1] = l4.y; loq[j + 2] = l4.z; loq[j + 3] = l4.w;
                        hiq[j] = h4.x; hiq[j + 1] = h4.y; hiq[j + 2] = h4.z; hiq[j + 3] = h4.w;
                    }
                    // (unused tiles: both thresholds +inf, never counted for finite moduli; their
                    // near bits are not stored)
                    int kb = 0, ka = 0;
                    unsigned long long near[kFarTiles];
#pragma unroll
                    for (int j = 0; j < kFarTiles; ++j) {
                        const bool below = frb <= loq[j], above = frs >= hiq[j];
                        kb += below ? 0 : 1;
                        ka += above ? 1 : 0;
                        near[j] = __builtin_amdgcn_ballot_w64(valid && !below && !above);
                    }
                    if (lane == 0) {   // the block's two mask words of every used tile
#pragma unroll
                        for (int j = 0; j < kFarTiles; ++j)
                            if ((used >> j) & 1u)
                                *reinterpret_cast<uint2 *>(mrow + static_cast<size_t>(j) * A.far_words + 2 * blk) =
                                    make_uint2(static_cast<unsigned int>(near[j]), static_cast<unsigned int>(near[j] >> 32));
                    }
                    // below: entry kb (< nv), series m_k; above: entry ka (> 0), series n_k.
                    // A thread whose entry changes first adds its running sums to the block's
                    // array; lanes with no share carry zero coefficients.
                    const bool hasB = valid && kb < nv, hasA = valid && ka > 0 && ka <= nv;
                    const bool swB = hasB && kb != cbB, swA = hasA && ka != cbA;
                    if (__builtin_amdgcn_ballot_w64(swB)) {
                        far_flush(sh.dB[wave], swB && cbB >= 0, cbB, accB);
#pragma unroll
                        for (int k = 0; k < kFarTerms; ++k) accB[k] = swB ? 0.0 : accB[k];
                        cbB = swB ? kb : cbB;
                    }
                    if (__builtin_amdgcn_ballot_w64(swA)) {
                        far_flush(sh.dA[wave], swA && cbA >= 0, cbA, accA);
#pragma unroll
                        for (int k = 0; k < kFarTerms; ++k) accA[k] = swA ? 0.0 : accA[k];
                        cbA = swA ? ka : cbA;
                    }
                    {
                        double a = hasB ? c.a : 0.0, cc = hasB ? c.c : 0.0;
                        double Ds2 = hasB ? 2.0 * Ds : 0.0, p0 = hasB ? P0 : 0.0;
                        // (the series start after the flushes: their terms are not held
                        // live across them)
                        asm volatile("" : "+v"(a), "+v"(cc), "+v"(Ds2), "+v"(p0));
                        double m0 = a, m1 = fma(Ds2, a, cc);
                        accB[0] += m0;
                        accB[1] += m1;
#pragma unroll
                        for (int k = 2; k < kFarTerms; ++k) {
                            const double m2 = fma(Ds2, m1, -p0 * m0);
                            accB[k] += m2;
                            m0 = m1;
                            m1 = m2;
                        }
                    }
                    {
                        double a = hasA ? c.a : 0.0, cc = hasA ? c.c : 0.0;
                        double Ds2 = hasA ? 2.0 * Ds : 0.0, iP = hasA ? recip(P0) : 0.0;
                        asm volatile("" : "+v"(a), "+v"(cc), "+v"(Ds2), "+v"(iP));
                        double n0 = cc * iP, n1 = fma(Ds2, n0, a) * iP;
                        accA[0] += n0;
                        accA[1] += n1;
#pragma unroll
                        for (int k = 2; k < kFarTerms; ++k) {
                            const double n2 = fma(Ds2, n1, -n0) * iP;
                            accA[k] += n2;
                            n0 = n1;
                            n1 = n2;
                        }
                    }
                }
                far_flush(sh.dB[wave], cbB >= 0, cbB, accB);
                far_flush(sh.dA[wave], cbA >= 0, cbA, accA);
                __syncthreads();
                // moments of each used tile: prefix sums of the below array up to its rank
                // by q lo, suffix sums of the above array past its rank by hi / q
                const int ss = kSegFarSet[SEG] + (inv ? v : 0);
                for (int e = tid; e < kFarTiles * kFarTerms; e += kThreads) {
                    const int j = e / kFarTerms, k = e % kFarTerms;
                    if (!((used >> j) & 1u)) continue;
                    const int pb = tile_rank<F32>(sh, used, j, rv, false), pa = tile_rank<F32>(sh, used, j, rv, true);
                    double sb = 0.0, sa = 0.0;
                    for (int w = 0; w < kFarWaves; ++w) {
                        for (int p = 0; p <= pb; ++p) sb += sh.dB[w][p][k];
                        for (int p = pa + 1; p <= nv; ++p) sa += sh.dA[w][p][k];
                    }
                    sh.mom[j][ss * 2 * kFarTerms + k] += sb;
                    sh.mom[j][ss * 2 * kFarTerms + kFarTerms + k] += sa;
                }
                __syncthreads();
                for (int e = tid; e < kFarWaves * (kFarTiles + 1) * kFarTerms; e += kThreads) {
                    (&sh.dB[0][0][0])[e] = 0.0;
                    (&sh.dA[0][0][0])[e] = 0.0;
                }
                __syncthreads();
            }
        });
    }
    for (int e = tid; e < kFarTiles * kFarMom; e += kThreads) {
        const int jj = e / kFarMom, r = e % kFarMom;
        const int t = g * kFarTiles + jj;
        if (t < A.tiles_total)
            A.far_mom[((static_cast<size_t>(layer) * nsplit + part) * A.tiles_total + t) * kFarMom + r] = sh.mom[jj][r];
    }
    // the h2o base term of this part's lines (every group derives them; group 0 writes)
    for (int m = 32; m > 0; m >>= 1) base += __shfl_xor(base, m);
    if (lane == 0) sh.bsum[wave] = base;
    __syncthreads();
    if (tid == 0 && g == 0) {
        double b = 0.0;
        for (int w = 0; w < kThreads / 64; ++w) b += sh.bsum[w];
        A.far_base[static_cast<size_t>(part) * A.nl + layer] = b;
    }
}

// ---- pass 2: near lines summed per tile, plus the series ----
//
// A near line is summed term by term only at the columns it is close to.  A term is analytic in
// f but for its poles +-sqrt(p), so over an interval of columns [lo, hi] that lies well away from
// them it is its Chebyshev interpolant on n nodes to rho^-n, rho the Bernstein ellipse (foci lo
// and hi) through the nearest pole: n values stand for all the interval's columns.  Lines outside
// rho are taken at nodes.  The rate alone does not give the error: a narrow line's two conjugate poles
// all but cancel (a near-double pole, n rho^-n), and its value at a far column is up to 13 times less
// than at the interval's near end.  For lines of every form with their pole on the ellipse, the worst
// error relative to the line's own value at the column, and to its largest in the interval:
//   16 nodes  rho 3.2: 3.5e-6, 2.5e-7   4.0: 8.7e-8, 1.2e-8   4.2: 4.6e-8, 6.3e-9
//   32 nodes  rho 3.2: 4.2e-14, 4e-15   3.6: 1.0e-15, 1.2e-16
// FP32 mode takes 16 nodes outside 4.2 (under one FP32 rounding, 6e-8), FP64 mode 32 outside 3.6 (the
// roundings of an FP64 term).
//
// A node's value reaches every column of its interval, so the node sums are FP64 in FP32 mode too:
// FP32 ones left tables 7 % (rms over 90 requests; at worst 25 %) further from FP64 than sums at
// every column, FP64 ones 6 % nearer.  At a leaf's columns FP32 mode sums as sum_staged_f32 does.
//
// The tile's columns form a binary tree of intervals (whole tile, halves, ... down to leaves of 32
// columns, 64 in FP64 mode).  A batch of 64 listed lines (neighbours in frequency, so they mostly
// agree) takes the largest intervals that all of its lines are outside the ellipse of, at their
// nodes, and a leaf that some line is close to at its columns.  Lanes are the points of one interval
// times groups of lines: 4 groups at 16 nodes, 2 at 32 points.  The sums stay per interval until the
// slot's last line; then their Chebyshev coefficients are formed and each column adds its ancestors'
// series.  Every column of every listed line against this, the pass alone: 400 layers x 512 columns x
// 11000 lines 331 -> 243 us (FP32), 812 -> 342 (FP64); 800 x 1024 x 26000 1517 -> 1171, 4195 -> 1882;
// 600 x 1000 x 11000 FP64 1569 -> 639; 300 x 201 FP64 421 -> 237.  (FP32 node sums outside rho = 3.2
// took 208 and 1067 us in FP32 mode.)  It is held at four wavefronts per SIMD (about 100 B of scratch a
// lane): 800 x 1024 x 26000, FP32, the whole request 2.85 ms with three, 2.64-2.78 with four.
template <bool F32>
__host__ __device__ constexpr double node_rho() { return F32 ? 4.2 : 3.6; }

template <int K, bool F32>
struct NearTree {
    static constexpr int nodes = F32 ? 16 : 32;
    static constexpr int width = F32 ? 32 : 64;         // columns of a leaf
    static constexpr int leaves = 64 * K / width;
    static constexpr int intervals = 2 * leaves;        // heap order: 1 the tile, 2i and 2i + 1 its halves
    static constexpr int node_groups = 64 / nodes, col_groups = 64 / width;   // line groups
};

// cos(j pi / 64), j = 0..127
constexpr int kCosTab = 128;
__constant__ double kCos64[kCosTab] = {
    1.0, 0.9987954562051724, 0.9951847266721969, 0.989176509964781,
    0.9807852804032304, 0.970031253194544, 0.9569403357322088, 0.9415440651830208,
    0.9238795325112867, 0.9039892931234433, 0.881921264348355, 0.8577286100002721,
    0.8314696123025452, 0.8032075314806449, 0.773010453362737, 0.7409511253549591,
    0.7071067811865476, 0.6715589548470184, 0.6343932841636455, 0.5956993044924334,
    0.5555702330196022, 0.5141027441932218, 0.47139673682599764, 0.4275550934302821,
    0.3826834323650898, 0.33688985339222005, 0.2902846772544624, 0.2429801799032639,
    0.19509032201612828, 0.14673047445536175, 0.0980171403295606, 0.049067674327418015,
    0.0, -0.049067674327418015, -0.0980171403295606, -0.14673047445536175,
    -0.19509032201612828, -0.2429801799032639, -0.2902846772544624, -0.33688985339222005,
    -0.3826834323650898, -0.4275550934302821, -0.47139673682599764, -0.5141027441932218,
    -0.5555702330196022, -0.5956993044924334, -0.6343932841636455, -0.6715589548470184,
    -0.7071067811865476, -0.7409511253549591, -0.773010453362737, -0.8032075314806449,
    -0.8314696123025452, -0.8577286100002721, -0.881921264348355, -0.9039892931234433,
    -0.9238795325112867, -0.9415440651830208, -0.9569403357322088, -0.970031253194544,
    -0.9807852804032304, -0.989176509964781, -0.9951847266721969, -0.9987954562051724,
    -1.0, -0.9987954562051724, -0.9951847266721969, -0.989176509964781,
    -0.9807852804032304, -0.970031253194544, -0.9569403357322088, -0.9415440651830208,
    -0.9238795325112867, -0.9039892931234433, -0.881921264348355, -0.8577286100002721,
    -0.8314696123025452, -0.8032075314806449, -0.773010453362737, -0.7409511253549591,
    -0.7071067811865476, -0.6715589548470184, -0.6343932841636455, -0.5956993044924334,
    -0.5555702330196022, -0.5141027441932218, -0.47139673682599764, -0.4275550934302821,
    -0.3826834323650898, -0.33688985339222005, -0.2902846772544624, -0.2429801799032639,
    -0.19509032201612828, -0.14673047445536175, -0.0980171403295606, -0.049067674327418015,
    0.0, 0.049067674327418015, 0.0980171403295606, 0.14673047445536175,
    0.19509032201612828, 0.2429801799032639, 0.2902846772544624, 0.33688985339222005,
    0.3826834323650898, 0.4275550934302821, 0.47139673682599764, 0.5141027441932218,
    0.5555702330196022, 0.5956993044924334, 0.6343932841636455, 0.6715589548470184,
    0.7071067811865476, 0.7409511253549591, 0.773010453362737, 0.8032075314806449,
    0.8314696123025452, 0.8577286100002721, 0.881921264348355, 0.9039892931234433,
    0.9238795325112867, 0.9415440651830208, 0.9569403357322088, 0.970031253194544,
    0.9807852804032304, 0.989176509964781, 0.9951847266721969, 0.9987954562051724,
};

// one wavefront's staged batch of kWaveBatch near lines
constexpr int kWaveBatch = 64;
struct WaveStage {
    alignas(16) double D[kWaveBatch];    // Ds
    alignas(16) double h[kWaveBatch];
    alignas(16) double a[kWaveBatch];    // a, c (scaled)
    alignas(16) double c[kWaveBatch];
    alignas(16) float2 ac[kWaveBatch];   // a, c and Ds, h rounded to FP32
    alignas(16) float2 dh[kWaveBatch];
};

// FP64 mode: the (D, a, c, g, G) of the direct FP64 sums
struct WaveStage64 {
    alignas(16) double D[kWaveBatch], a[kWaveBatch], c[kWaveBatch], g[kWaveBatch], G[kWaveBatch];
};

// An interval of the tile's columns in f, of one range (kFarRanges); hi < lo: no columns
struct NearInterval {
    double c, r;          // centre, half width
    float lo, hi, thr;    // thr: the least |z - lo| + |z - hi| of a pole outside the ellipse (NaN: none is)
};

template <int K, bool F32>
struct NearShared {
    using Tree = NearTree<K, F32>;
    std::conditional_t<F32, WaveStage, WaveStage64> st[kThreads / 64];
    // the wavefronts' sums at the intervals' nodes and at the columns
    double node[kThreads / 64][Tree::intervals][Tree::nodes];
    double column[kThreads / 64][64 * K];
    union {
        unsigned short list[kListWords * 32];   // a window's near lines
        double cheb[2][Tree::intervals][Tree::nodes];   // node sums, Chebyshev coefficients
    };
    double far[kFarMom];
    NearInterval iv[kFarRanges][Tree::intervals];
    double cosines[kCosTab];
    int wsum[kThreads / 64];
    int used;                        // some wavefront has added to node or column
    alignas(16) double prep[2][8];   // the segment's coefficient sets (read from LDS while deriving)
    double scale[2];                 // and their FP32 weight scales
};

// sum of the far-line series of one moment set at x
__device__ inline double far_eval(const double *mom, double x) {
    double below = 0.0;
    if (x > 0.0) {
        const double u = 1.0 / x;
        double s = mom[kFarTerms - 1];
#pragma unroll
        for (int k = kFarTerms - 2; k >= 0; --k) s = fma(s, u, mom[k]);
        below = s * u;
    }
    const double *n = mom + kFarTerms;
    double s = n[kFarTerms - 1];
#pragma unroll
    for (int k = kFarTerms - 2; k >= 0; --k) s = fma(s, x, n[k]);
    return below + s;
}

// A listed line's coefficients for the near sums, derived from its catalogue row as pass 1
// derives them, with the segment's coefficient sets read from LDS: FP32 mode (Ds, h, a s, c s),
// FP64 mode (D, a, c, g, G)
template <class Prep, int NC>
__device__ __forceinline__ CoefT<double> near_coef(const DevBlock &B, int i, int v, const double (&prep)[2][8]) {
    LineRow<NC> row;
    row.load(B, i);
    double unused = 0.0;
    return seg_coef(*reinterpret_cast<const Prep *>(prep[0]), *reinterpret_cast<const Prep *>(prep[1]), v, row, i,
                    unused);
}

template <bool F32>
__device__ __forceinline__ void derive_near(int seg, int v, const DevBlock &B, int i, const double (&prep)[2][8],
                                            double sv, double (&c5)[5]) {
    CoefT<double> c;
    switch (seg) {
        case 0: c = near_coef<H2oPrep<double>, kNumCols[RBX_LINES_H2O]>(B, i, v, prep); break;
        case 1: c = near_coef<H2sPrep<double>, kNumCols[RBX_LINES_H2S]>(B, i, v, prep); break;
        case 2: c = near_coef<InvPrep<double>, kNumCols[RBX_LINES_NH3_INV]>(B, i, v, prep); break;
        case 3: c = near_coef<RotPrep<double>, kNumCols[RBX_LINES_NH3_ROT]>(B, i, v, prep); break;
        case 4: c = near_coef<V2Prep<double>, kNumCols[RBX_LINES_NH3_V2]>(B, i, v, prep); break;
        default: c = near_coef<Ph3Prep<double>, kNumCols[RBX_LINES_PH3]>(B, i, v, prep); break;
    }
    if constexpr (F32) {
        shifted_denominator(c, c5[0], c5[1]);
        c5[2] = c.a * sv;
        c5[3] = c.c * sv;
    } else {
        c5[0] = c.D;
        c5[1] = c.a;
        c5[2] = c.c;
        c5[3] = c.g;
        c5[4] = c.G;
    }
}

// v summed over the wavefront's `G` line groups (lane bits 5, then 4), in every lane
template <int G>
__device__ __forceinline__ double group_sum(double v) {
    using Words = unsigned int __attribute__((ext_vector_type(2)));
    auto add = [](double y, auto &&swap) {
        const Words w = __builtin_bit_cast(Words, y);
        const auto lo = swap(w.x), hi = swap(w.y);
        return __builtin_bit_cast(double, Words{lo[0], hi[0]}) + __builtin_bit_cast(double, Words{lo[1], hi[1]});
    };
    if constexpr (G >= 4) v = add(v, [](unsigned int q) { return __builtin_amdgcn_permlane16_swap(q, q, false, false); });
    if constexpr (G >= 2) v = add(v, [](unsigned int q) { return __builtin_amdgcn_permlane32_swap(q, q, false, false); });
    return v;
}

// The pole in f nearest the positive axis of (x - Ds)^2 + h: sqrt(Ds + i sqrt(h)) for a complex
// pair; for h < 0 (a coupling or width beyond the centre: both poles real and negative) i times the
// root of the smaller modulus.  Anything else gives NaN, which is close to every interval.
__device__ __forceinline__ float2 pole_in_f(double Ds, double h) {
    const float d = static_cast<float>(Ds), q = __builtin_amdgcn_sqrtf(fabsf(static_cast<float>(h)));
    if (h >= 0.0) {
        const float m = __builtin_amdgcn_sqrtf(static_cast<float>(fma(Ds, Ds, h)));
        const float big = __builtin_amdgcn_sqrtf(0.5f * (m + fabsf(d)));
        const float small = 0.5f * q / big;
        return d >= 0.0f ? make_float2(big, small) : make_float2(small, big);
    }
    return make_float2(0.0f, d < 0.0f && q <= -d ? __builtin_amdgcn_sqrtf(-d - q) : NAN);
}

__device__ __forceinline__ bool outside(const float2 &z, const NearInterval &I) {
    const float a = z.x - I.lo, b = z.x - I.hi, y2 = z.y * z.y;
    return __builtin_amdgcn_sqrtf(fmaf(a, a, y2)) + __builtin_amdgcn_sqrtf(fmaf(b, b, y2)) >= I.thr;
}

// Sum of the staged lines' terms at this lane's point x, over the pairs of lines g, g + G, ... of
// the batch's first `npairs` (a multiple of 4 G), two lines over one denominator: in FP64 from
// (Ds, h, a, c) ...
template <int G>
__device__ __forceinline__ double sum_pairs(const WaveStage &st, int g, int npairs, double x) {
    double acc = 0.0;
#pragma unroll 2
    for (int p = g; p < npairs; p += G) {
        const double2 D = reinterpret_cast<const double2 *>(st.D)[p], h = reinterpret_cast<const double2 *>(st.h)[p];
        const double2 a = reinterpret_cast<const double2 *>(st.a)[p], c = reinterpret_cast<const double2 *>(st.c)[p];
        const double d1 = x - D.x, d2 = x - D.y;
        const double n1 = fma(a.x, x, c.x), n2 = fma(a.y, x, c.y);
        const double e1 = fma(d1, d1, h.x), e2 = fma(d2, d2, h.y);
        acc += fma(n1, e2, n2 * e1) * recip(e1 * e2);
    }
    return acc;
}

// ... and from (D, a, c, g, G), the terms of sum_staged_f64
template <int G>
__device__ __forceinline__ double sum_pairs(const WaveStage64 &st, int g, int npairs, double x) {
    double acc = 0.0;
#pragma unroll 2
    for (int p = g; p < npairs; p += G) {
        const double2 D = reinterpret_cast<const double2 *>(st.D)[p], a = reinterpret_cast<const double2 *>(st.a)[p];
        const double2 c = reinterpret_cast<const double2 *>(st.c)[p], gg = reinterpret_cast<const double2 *>(st.g)[p];
        const double2 GG = reinterpret_cast<const double2 *>(st.G)[p];
        const double d1 = x - D.x, d2 = x - D.y;
        const double n1 = fma(a.x, x, c.x), n2 = fma(a.y, x, c.y);
        const double e1 = fma(d1, d1, fma(gg.x, x, GG.x)), e2 = fma(d2, d2, fma(gg.y, x, GG.y));
        acc += fma(n1, e2, n2 * e1) * recip(e1 * e2);
    }
    return acc;
}

// The same at a column in FP32 mode (sum_staged_f32), blocks of 8 lines in FP32.  `fast`: bit j = lines
// [8 j, 8 j + 8) are FP32-safe for the tile's columns; the others form their denominators in FP64.
template <int G>
__device__ __forceinline__ double sum_pairs_f32(const WaveStage &st, int g, int npairs, double x, unsigned int fast) {
    const float xf = static_cast<float>(x);
    constexpr unsigned int kAll = (1u << G) - 1u;
    double acc = 0.0;
    for (int p0 = 0; p0 < npairs; p0 += 4 * G) {
        float p = 0.0f;
        if (((fast >> (p0 / 4)) & kAll) == kAll) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const float4 dp = reinterpret_cast<const float4 *>(st.dh)[p0 + u * G + g];
                const float4 qp = reinterpret_cast<const float4 *>(st.ac)[p0 + u * G + g];
                const float d1 = xf - dp.x, d2 = xf - dp.z;
                const float e1 = fmaf(d1, d1, dp.y), e2 = fmaf(d2, d2, dp.w);
                const float n1 = fmaf(qp.x, xf, qp.y), n2 = fmaf(qp.z, xf, qp.w);
                p = fmaf(fmaf(n2, e1, n1 * e2), __builtin_amdgcn_rcpf(e1 * e2), p);
            }
        } else {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const double2 Dp = reinterpret_cast<const double2 *>(st.D)[p0 + u * G + g];
                const double2 hp = reinterpret_cast<const double2 *>(st.h)[p0 + u * G + g];
                const float4 qp = reinterpret_cast<const float4 *>(st.ac)[p0 + u * G + g];
                const double d1 = x - Dp.x, d2 = x - Dp.y;
                const float e1 = static_cast<float>(fma(d1, d1, hp.x)), e2 = static_cast<float>(fma(d2, d2, hp.y));
                const float n1 = fmaf(qp.x, xf, qp.y), n2 = fmaf(qp.z, xf, qp.w);
                p = fmaf(fmaf(n2, e1, n1 * e2), __builtin_amdgcn_rcpf(e1 * e2), p);
            }
        }
        acc += static_cast<double>(p);
    }
    return acc;
}

// A batch's staged lines added at the tree's points: this lane's line has pole z (`line` false:
// padding, a zero term); `fast` as for sum_pairs_f32; columns' x of the leaves from `colx`.
template <int K, bool F32, class ColX>
__device__ __forceinline__ void sum_tree(NearShared<K, F32> &sh, int rv, bool line, const float2 &z, unsigned int fast,
                                         int count, double inv_scale, const ColX &colx) {
    using Tree = NearTree<K, F32>;
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    const auto &st = sh.st[wave];
    const double node = sh.cosines[(2 * (lane % Tree::nodes) + 1) * (kCosTab / 4 / Tree::nodes)];
    unsigned int pending = 2u;
#pragma unroll 1
    for (int i = 1; i < Tree::intervals; ++i) {
        if (!((pending >> i) & 1u)) continue;
        const NearInterval I = sh.iv[rv][i];
        if (!(I.lo <= I.hi)) continue;   // no columns
        const bool nodes = __all(!line || outside(z, I));
        if (!nodes && i < Tree::leaves) {
            pending |= 3u << (2 * i);
            continue;
        }
        if (nodes) {
            constexpr int G = Tree::node_groups;
            const double f = fma(I.r, node, I.c);
            const double s = group_sum<G>(sum_pairs<G>(st, lane / Tree::nodes, (count + 8 * G - 1) / (8 * G) * (4 * G), f * f));
            double &v = sh.node[wave][i][lane % Tree::nodes];
            if (lane < Tree::nodes) v = fma(s, inv_scale, v);
        } else {
            constexpr int G = Tree::col_groups;
            const int k = (i - Tree::leaves) * Tree::width + lane % Tree::width;
            const int npairs = (count + 8 * G - 1) / (8 * G) * (4 * G);
            double s;
            if constexpr (F32)
                s = sum_pairs_f32<G>(st, lane / Tree::width, npairs, colx(k), fast);
            else
                s = sum_pairs<G>(st, lane / Tree::width, npairs, colx(k));
            s = group_sum<G>(s);
            double &v = sh.column[wave][k];
            if (lane < Tree::width) v = fma(s, inv_scale, v);
        }
    }
}

// near lines of one segment and coefficient set v, listed from the tile's mask words; each
// wavefront sums its own batches of kWaveBatch listed lines (batches w, w + 4, ...), staged in its
// own LDS.
template <int K, bool F32, class Derive, class ColX>
__device__ void near_sum(int n, const Derive &derive, int rv, const unsigned int *mask, int nwords, double inv_scale,
                         const ColX &colx, NearShared<K, F32> &sh) {
    const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
    auto &st = sh.st[wave];
    for (int w0 = 0; w0 < nwords; w0 += kListWords) {
        const int wi = w0 + tid;
        const unsigned int bits = (tid < kListWords && wi < nwords) ? mask[wi] : 0u;
        const int cnt = __popc(bits);
        int incl = cnt;
#pragma unroll
        for (int m = 1; m < 64; m <<= 1) {
            const int y = __shfl_up(incl, m);
            if (lane >= m) incl += y;
        }
        if (lane == 63) sh.wsum[wave] = incl;
        __syncthreads();
        int pos = incl - cnt, total = 0;
#pragma unroll
        for (int w = 0; w < kThreads / 64; ++w) {
            if (w < wave) pos += sh.wsum[w];
            total += sh.wsum[w];
        }
        for (unsigned int b = bits; b != 0u; b &= b - 1u)
            sh.list[pos++] = static_cast<unsigned short>(tid * 32 + __builtin_ctz(b));
        if (total > 0 && tid == 0) sh.used = 1;
        __syncthreads();
        // listed line e's coefficients, derived from its catalogue row when its batch is
        // staged (past the list: a zero term): FP32 mode (Ds, h, a s, c s), FP64 mode (D, a, c, g, G)
        const int nb = (total + kWaveBatch - 1) / kWaveBatch;
        for (int b = wave; b < nb; b += kThreads / 64) {
            const int e = b * kWaveBatch + lane;
            const int i = e < total ? w0 * 32 + sh.list[e] : n;
            double c5[5] = {0.0, F32 ? 1.0 : 0.0, 0.0, 0.0, 1.0};
            if (i < n) derive(i, c5);
            double Ds = c5[0], h = c5[1];
            unsigned int fast = 0u;
            wave_sync();   // (the batch before has been summed)
            if constexpr (F32) {
                const double lo = sh.iv[rv][1].lo, hi = sh.iv[rv][1].hi;
                st.D[lane] = Ds;
                st.h[lane] = h;
                st.a[lane] = c5[2];
                st.c[lane] = c5[3];
                st.ac[lane] = make_float2(static_cast<float>(c5[2]), static_cast<float>(c5[3]));
                st.dh[lane] = make_float2(static_cast<float>(Ds), static_cast<float>(h));
                fast = full_chunks(__ballot(lo >= 0.0 && fp32_safe(Ds, h, lo * lo, hi * hi)));
            } else {
                st.D[lane] = c5[0];
                st.a[lane] = c5[1];
                st.c[lane] = c5[2];
                st.g[lane] = c5[3];
                st.G[lane] = c5[4];
                shifted_denominator(CoefT<double>{c5[0], c5[1], c5[2], c5[3], c5[4]}, Ds, h);
            }
            wave_sync();
            sum_tree<K, F32>(sh, rv, i < n, pole_in_f(Ds, h), fast, min(kWaveBatch, total - b * kWaveBatch), inv_scale,
                             colx);
        }
        __syncthreads();   // every wavefront is done with this window's list
    }
}

// The sums at the tree's points brought to column `tid` (threads below the tile's width): the
// wavefronts' and line groups' sums in order, the intervals' Chebyshev coefficients, and the series
// of the column's ancestors at its f.  Clears the sums; called by the whole block.
template <int K, bool F32>
__device__ double tree_to_column(NearShared<K, F32> &sh, int rv, double f) {
    using Tree = NearTree<K, F32>;
    const int tid = threadIdx.x;
    __syncthreads();
    if (!sh.used) return 0.0;   // (the same for every thread; nothing has been added)
    const int i0 = tid / Tree::nodes, k0 = tid % Tree::nodes;
    if (i0 >= 1 && i0 < Tree::intervals) {
        double s = 0.0;
        for (int w = 0; w < kThreads / 64; ++w) s += sh.node[w][i0][k0];
        sh.cheb[0][i0][k0] = s;
    }
    __syncthreads();
    if (i0 >= 1 && i0 < Tree::intervals) {
        double s = 0.0;
#pragma unroll
        for (int k = 0; k < Tree::nodes; ++k)
            s = fma(sh.cheb[0][i0][k], sh.cosines[(k0 * (2 * k + 1) * (kCosTab / 4 / Tree::nodes)) % kCosTab], s);
        sh.cheb[1][i0][k0] = s * ((k0 == 0 ? 1.0 : 2.0) / Tree::nodes);
    }
    __syncthreads();
    double out = 0.0;
    if (tid < 64 * K) {
        const int leaf = tid / Tree::width;
        for (int w = 0; w < kThreads / 64; ++w) out += sh.column[w][tid];
        for (int i = Tree::leaves + leaf; i >= 1; i >>= 1) {
            const NearInterval &I = sh.iv[rv][i];
            if (!(I.thr >= 0.0f)) continue;   // no nodes taken (c and r may not be finite)
            const double u = I.r > 0.0 ? (f - I.c) / I.r : 0.0, u2 = 2.0 * u;
            double b1 = 0.0, b2 = 0.0;   // Clenshaw
#pragma unroll
            for (int m = Tree::nodes - 1; m >= 1; --m) {
                const double b0 = fma(u2, b1, sh.cheb[1][i][m] - b2);
                b2 = b1;
                b1 = b0;
            }
            out += fma(u, b1, sh.cheb[1][i][0] - b2);
        }
    }
    __syncthreads();
    for (int e = tid; e < (kThreads / 64) * Tree::intervals * Tree::nodes; e += kThreads) (&sh.node[0][0][0])[e] = 0.0;
    for (int e = tid; e < (kThreads / 64) * 64 * K; e += kThreads) (&sh.column[0][0])[e] = 0.0;
    if (tid == 0) sh.used = 0;
    __syncthreads();
    return out;
}

template <int K, bool F32>
__global__ __launch_bounds__(kThreads, 4) void alpha_near_kernel(AlphaArgs args) {
#if defined(__HIP_DEVICE_COMPILE__)
    const AlphaArgs &A = *reinterpret_cast<const AlphaArgs *>(__builtin_amdgcn_kernarg_segment_ptr());
#else
    const AlphaArgs &A = args;   // (host pass: never run)
#endif
    using Tree = NearTree<K, F32>;
    __shared__ NearShared<K, F32> sh;
    // layer fastest: blocks are dealt to the XCDs in turn, so each XCD gets every tile (the
    // tiles' near fractions differ several-fold) rather than one tile of every layer.  Last
    // tile first: requests run low to high frequency and line lists grow denser with frequency,
    // so the heavy tiles start first and the light ones fill the tail of the grid (800 layers
    // x 1024 frequencies: step 3.92 -> 3.73 ms).
    const int layer = blockIdx.x % A.nl, tile = A.tiles_total - 1 - static_cast<int>(blockIdx.x / A.nl);
    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int nsplit = A.far_split;
    const LayerT<double> L = layer_of(A, layer);
    int c0, c1;
    tile_cols(A, tile, c0, c1);
    const int tsets = tile_sets(A, c0, c1);
    const bool mixed = tsets == 3;   // the tile straddles the switch between the inversion sets

    // thread tid owns column c0 + tid
    const int col = c0 + tid;
    const bool ok = tid < 64 * K && col < A.nf;
    const int cc = min(col, A.nf - 1);
    const int set = cc < A.nf_low ? 0 : 1;
    const double f = A.freq[cc], fn = A.freq_nh3 ? A.freq_nh3[cc] : f;

    // the tree's intervals: wavefront v the range v, leaves first (LDS: lo and hi in c and r)
    static_assert(kFarRanges == kThreads / 64, "a wavefront per range");
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int cl = c0 + k * 64 + lane;
        const bool in = cl < c1 && (wave < 2 || (cl < A.nf_low ? 2 : 3) == wave);
        const int ccl = min(cl, A.nf - 1);
        const double fl = wave > 0 && A.freq_nh3 ? A.freq_nh3[ccl] : A.freq[ccl];
        double lo = in ? fl : INFINITY, hi = in ? fl : -INFINITY;
#pragma unroll
        for (int m = Tree::width / 2; m > 0; m >>= 1) {
            lo = fmin(lo, __shfl_xor(lo, m));
            hi = fmax(hi, __shfl_xor(hi, m));
        }
        if (lane % Tree::width == 0) {
            NearInterval &I = sh.iv[wave][Tree::leaves + k * Tree::col_groups + lane / Tree::width];
            I.c = lo;
            I.r = hi;
        }
    }
    wave_sync();
#pragma unroll
    for (int lev = Tree::leaves / 2; lev >= 1; lev /= 2) {
        if (lane >= lev && lane < 2 * lev) {
            const NearInterval a = sh.iv[wave][2 * lane], b = sh.iv[wave][2 * lane + 1];
            sh.iv[wave][lane].c = fmin(a.c, b.c);
            sh.iv[wave][lane].r = fmax(a.r, b.r);
        }
        wave_sync();
    }
    if (lane >= 1 && lane < Tree::intervals) {
        NearInterval &I = sh.iv[wave][lane];
        const double lo = I.c, hi = I.r;
        I.lo = static_cast<float>(lo);
        I.hi = static_cast<float>(hi);
        I.c = 0.5 * (lo + hi);
        I.r = 0.5 * (hi - lo);
        // The margin covers the FP32 roundings of lo, hi and the poles.  No nodes (thr NaN: no pole is
        // outside) where f < 0, or past where the FP32 distances' squares overflow (f infinite).  A
        // node's f is rounded to 2^-53 c, which moves a term by up to about 2^-53 c / r of itself:
        // FP64 mode takes no nodes in narrow intervals.
        const bool use = lo >= 0.0 && hi < 1.0e15 && (F32 || 64.0 * I.r >= I.c);
        I.thr = use ? static_cast<float>(I.r * (node_rho<F32>() + 1.0 / node_rho<F32>()) + 1.0e-6 * hi) : NAN;
    }
    for (int e = tid; e < kFarMom; e += kThreads) {
        double s = 0.0;
        for (int p = 0; p < nsplit; ++p)
            s += A.far_mom[((static_cast<size_t>(layer) * nsplit + p) * A.tiles_total + tile) * kFarMom + e];
        sh.far[e] = s;
    }
    if (tid < kCosTab) sh.cosines[tid] = kCos64[tid];
    for (int e = tid; e < (kThreads / 64) * Tree::intervals * Tree::nodes; e += kThreads) (&sh.node[0][0][0])[e] = 0.0;
    for (int e = tid; e < (kThreads / 64) * 64 * K; e += kThreads) (&sh.column[0][0])[e] = 0.0;
    if (tid == 0) sh.used = 0;
    if (tile == 0 && tid == 0) {
        double b = 0.0;
        for (int p = 0; p < nsplit; ++p) b += A.far_base[static_cast<size_t>(p) * A.nl + layer];
        A.ws_base[layer] = b;
    }
    __syncthreads();

    const LinePlan plan(A, L.P);
    const int touched = plan.slots(0, 1);
    const size_t plane = static_cast<size_t>(A.nl) * A.nf;
    const unsigned int *masks = A.near + (static_cast<size_t>(layer) * A.tiles_total + tile) * A.far_words;
    auto series = [&](int q) {
        const double x = f * f, xn = fn * fn;
        switch (q) {
            case kSlotH2o: return far_eval(sh.far + 0 * 2 * kFarTerms, x);
            case kSlotH2s: return far_eval(sh.far + 1 * 2 * kFarTerms, x);
            case kSlotNh3:
                return far_eval(sh.far + (2 + set) * 2 * kFarTerms, xn) + far_eval(sh.far + 4 * 2 * kFarTerms, xn);
            default: return far_eval(sh.far + 5 * 2 * kFarTerms, x);
        }
    };
    double acc = 0.0;   // column tid's sum of the current slot
    auto store = [&](int q) {
        if ((touched & (1 << q)) && ok)
            A.ws[static_cast<size_t>(q) * plane + static_cast<size_t>(layer) * A.nf + col] = acc + series(q);
        acc = 0.0;
    };
    for (int seg = 0; seg < kSegs; ++seg) {
        const bool inv = seg == 2;
        const int var = kSegVar[seg];
        if (plan.nr[seg] > 0) {
            // the segment's coefficient sets and weight scales go to LDS and are read there
            // while deriving (held in registers across the line sums they would crowd out the
            // sums' own)
            __syncthreads();   // (the previous segment's derivations are done)
            if (tid < kPrepWords) {
                const double w = A.far_prep[(static_cast<size_t>(layer) * kSegs + seg) * kPrepWords + tid];
                if (tid < 16)
                    sh.prep[tid / 8][tid % 8] = w;
                else
                    sh.scale[tid - 16] = w;
            }
            __syncthreads();
            const DevBlock &B = A.cat.blk[kSegKind[seg]];
            const int nwords = plan.nr[seg] * (kThreads / 32);
            auto colx = [&](int k) {
                const int ck = min(c0 + k, A.nf - 1);
                const double fk = var && A.freq_nh3 ? A.freq_nh3[ck] : A.freq[ck];
                return fk * fk;
            };
#pragma unroll 1
            for (int v = 0; v < 2; ++v) {
                if (inv ? !((tsets >> v) & 1) : v > 0) continue;
                const unsigned int *mk = masks + A.far_off[kSegStream[seg] + (inv ? v : 0)];
                const double sv = sh.scale[v];
                auto derive = [&](int i, double (&c5)[5]) { derive_near<F32>(seg, v, B, i, sh.prep, sv, c5); };
                const int rv = inv ? 2 + v : var;
                near_sum<K, F32>(B.n, derive, rv, mk, nwords, 1.0 / sv, colx, sh);   // (sv is a power of two)
                // of a tile of both sets only set v's columns, over their own intervals
                if (inv && mixed) {
                    const double s = tree_to_column<K, F32>(sh, rv, fn);
                    if (set == v) acc += s;
                }
            }
        }
        if (seg == 0 || seg == 1 || seg == 4 || seg == 5) {
            acc += tree_to_column<K, F32>(sh, var, var ? fn : f);
            store(seg == 0 ? kSlotH2o : seg == 1 ? kSlotH2s : seg == 4 ? kSlotNh3 : kSlotPh3);
        }
    }
}
