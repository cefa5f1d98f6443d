// Decode-time attention in one pass (included by attention.hip after interp.hpp).
//
// A decode step issues, per layer, q.K^T (at most 8 query rows per KV head after the GQA
// group is folded into rows), the soft-max program over the scores, and p.V.  Each of the
// three reads or writes the [rows, T] score matrix and the two products each stream the
// cache once from a launch of their own.  When the scores product is still lazy at the
// moment its soft-max becomes the left operand of p.V (see LazyMm), the three run here
// instead: a workgroup takes one KV head and one chunk of the T cached positions, computes
// its scores from K, runs the soft-max program on them with the chunk as the row (local
// maximum m_c, local sum l_c of exp(x - m_c)), multiplies the un-normalised weights with its
// chunk of V, and writes (m_c, l_c, o_c).  A second small kernel combines the chunks:
//     out = sum_c e^(m_c - g) o_c / sum_c e^(m_c - g) l_c,   g = max_c m_c,
// which is the soft-max-weighted sum written with another grouping of the same terms.
// The program is the compiled RowsSoftmaxCausal; its instructions before the row maximum
// (scale, causal mask) and between maximum and sum (subtract, exp) are evaluated by the
// same template code as in aot_rows_kernel, the final division is replaced by the combine.
// HBM-bound: K and V once (2 x 4 x T x head_dim bytes per KV head) + the chunk results.
#pragma once

#include <type_traits>

typedef float float4v __attribute__((ext_vector_type(4)));

// Leaf words of leaves FIRST.. of one work item (leaf 0 of the attention program has no memory).
template <class P, int VEC, int FIRST, int... L>
__device__ __forceinline__ void aot_load_from(const FusedArgs &a, const int64_t (&off)[P::nleaf + 1], uint32_t e,
                                              uint32_t (&v)[P::nleaf][VEC], std::integer_sequence<int, L...>) {
    (aot_load_leaf<P, VEC, FIRST + L>(a, off, e, v[FIRST + L]), ...);
}
template <class P, int FIRST>
__device__ __forceinline__ void aot_fetch_from(const FusedArgs &a, const int64_t (&base)[P::nleaf + 1], uint32_t it,
                                               LeafWords<P, 1> &w) {
    int64_t off[P::nleaf + 1];
#pragma unroll
    for (int l = 0; l < P::nleaf; l++) off[l] = base[l] + (int64_t)it * a.leaf[l].is;
    off[P::nleaf] = 0;
    aot_load_from<P, 1, FIRST>(a, off, it, w.v, std::make_integer_sequence<int, P::nleaf - FIRST>{});
}

// Sum over the 16 lanes of a DPP row (lanes 16i..16i+15), left in every lane of the row: four
// rotate-and-add steps inside the vector ALU instead of four trips through the LDS crossbar.
__device__ __forceinline__ float row16_sum(float v) {
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xF, 0xF, false)); // row_ror:8
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x124, 0xF, 0xF, false)); // row_ror:4
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x122, 0xF, 0xF, false)); // row_ror:2
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x121, 0xF, 0xF, false)); // row_ror:1
    return v;
}

struct AttnArgs {
    const uint32_t *Q, *Kc, *V;
    float *part_o;  // [batch][splits][M][hd]
    float *part_ml; // [batch][splits][M][2]
    uint32_t M, T, hd, splits, chunk;
    uint32_t nb;
    FastDiv groups; // decode, a workgroup per row: rows x parts of an entry
    // batch axes; decode: the slots behind nb hold axes of extent one
    uint32_t bd[kMaxBatchAxes];
    FastDiv bdiv[kMaxBatchAxes];
    int64_t q_bs[kMaxBatchAxes], k_bs[kMaxBatchAxes], v_bs[kMaxBatchAxes];
    int64_t p_rows[kMaxBatchAxes]; // decode: rows of the soft-max program per step of the axis
    int64_t q_sm; // stride between the query rows of a group
    int64_t k_st; // stride between cached positions of K (head_dim contiguous)
    int64_t v_st; // stride between cached positions of V (head_dim contiguous)
    // prefill only: the batch axes as p.V collapsed them (same number of entries, possibly another split)
    uint32_t nbv;
    uint32_t vbd[kMaxBatchAxes];
    FastDiv vbdiv[kMaxBatchAxes];
};

// q and the cache's newest row of K as the products left them (see OpenHeads): the kernels below apply the heads' RMS norm and the
// rotary embedding themselves, op for op as the launch that they save but for the order of the sum of squares, and store the results where
// that would have.  A wave finishes a row, behind the first loads of K, and the rows cross to the others through LDS.  The newest row's
// score is taken from there: the cache does not hold that row until the launch ends (what is loaded in its place is not used).
// head_norm_rope_finish_kernel takes 3.3 us and the hand-over behind it; here it hides behind K: Qwen3-0.6B's steps at 1050 positions
// (8 KV heads of 128, 2 query heads each) 7.41 us with finished heads, 7.48 so.  (Every wave finishing the rows for itself: the
// registers do not hold it all, 13.7.)
struct NoHeads {};
struct HeadRows { // of one product: HD columns a head, piece l of a row to lane l
    const float *src, *gamma, *cos, *sin;
    uint32_t n, n_bits, eps_bits, exp_bits; // n: columns of a row
};
struct RawHeads {
    HeadRows q, k;
    FastDiv heads; // KV heads: batch entry = sequence * heads + KV head
};
template <int LPT> struct OpenHead { // a wave's: a lane's piece of a row and the one that the embedding mixes it with, and the factors of both
    float4v x, other, gamma, gamma_other, cos, sin;
    __device__ __forceinline__ void load(const HeadRows &h, uint64_t row, uint32_t l) {
        const uint32_t l2 = l ^ (LPT / 2);
        auto piece = [](const float *p, uint32_t at) { return *reinterpret_cast<const float4v *>(p + at * 4); };
        x = piece(h.src + row, l);
        other = piece(h.src + row, l2);
        gamma = piece(h.gamma, l);
        gamma_other = piece(h.gamma, l2);
        cos = piece(h.cos, l);
        sin = piece(h.sin, l);
    }
    __device__ __forceinline__ float4v finish(const HeadRows &h, uint32_t l) const {
        float ss = row16_sum(fmaf(x[3], x[3], fmaf(x[2], x[2], fmaf(x[1], x[1], x[0] * x[0]))));
        if (LPT == 32) ss = asf(fold_rows(asu(ss), AddWords{}));
        const float r = norm_divisor(ss, h.n_bits, h.eps_bits, h.exp_bits);
        float4v v;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float own = x[j] / r * gamma[j], mixed = other[j] / r * gamma_other[j];
            v[j] = cos[j] * own + sin[j] * (l < LPT / 2 ? -mixed : mixed);
        }
        return v;
    }
};

// Operand offsets of batch entry b, and its first row in the soft-max program's [rows, T] space.  Two axes are read without a test (as a
// rule there are no more): a test in front of every axis is a trip to the argument block for every axis, a third of a microsecond each
// before the first load of K goes out.
__device__ __forceinline__ void entry_offsets(const AttnArgs &g, uint32_t b, int64_t &oq, int64_t &ok, int64_t &ov, uint32_t &row) {
    oq = ok = ov = 0;
    row = 0;
    auto axis = [&](const uint32_t d) {
        const uint32_t q = fastdiv(b, g.bdiv[d]), i = b - q * g.bd[d];
        b = q;
        oq += (int64_t)i * g.q_bs[d];
        ok += (int64_t)i * g.k_bs[d];
        ov += (int64_t)i * g.v_bs[d];
        row += i * (uint32_t)g.p_rows[d];
    };
    axis(0);
    axis(1);
    if (g.nb > 2)
        for (uint32_t d = 2; d < g.nb; d++) axis(d);
}
// the offsets of a row of that space in the program's leaves but the first, likewise
template <class P> __device__ __forceinline__ void leaf_offsets(const FusedArgs &a, uint32_t row, int64_t (&base)[P::nleaf + 1]) {
#pragma unroll
    for (int i = 0; i <= P::nleaf; i++) base[i] = 0;
    auto axis = [&](const uint32_t d) {
        const uint32_t q = fastdiv(row, a.g.odiv[d]), i = row - q * a.g.od[d];
        row = q;
#pragma unroll
        for (int lf = 1; lf < P::nleaf; lf++) base[lf] += (int64_t)i * a.leaf[lf].os[d];
    };
    axis(0);
    axis(1);
    if (a.g.nouter > 2)
        for (uint32_t d = 2; d < a.g.nouter; d++) axis(d);
}

constexpr int kAttnRows = 8;    // most query rows per KV head
constexpr int kAttnPasses = 8; // cached positions per lane group and workgroup
// most cached positions per workgroup: 128 for head_dim 64, 64 for head_dim 128
constexpr int attn_chunk_cap(int lpt) { return kAttnPasses * (kBlock / lpt); }

// LPT lanes share a cached position (head_dim / 4): 16 or 32.  Every lane first asks for all of
// its K and V pieces of the chunk (at most 2 x 8 sixteen-byte loads in flight), so the chunk
// costs one trip to memory; scores, soft-max and the weighted sum then run out of registers and LDS.
template <class P, int LPT>
__global__ __launch_bounds__(kBlock) void decode_attention_kernel(const AttnArgs g, const FusedArgs a) {
    constexpr int HD = LPT * 4;
    constexpr int TPB = kBlock / LPT; // positions per pass
    constexpr int CAP = attn_chunk_cap(LPT);
    constexpr int IPL = CAP / 64; // chunk positions per lane in the soft-max phase
    constexpr int ri0 = reduce_index<P>(0), ri1 = reduce_index<P>(1);
    constexpr int src0 = P::code[ri0][1], src1 = P::code[ri1][1];
    static_assert((P::code[ri0][0] & ~kInstrU32) == kRowMax && (P::code[ri1][0] & ~kInstrU32) == kRowSum,
                  "a soft-max: row maximum, then row sum");
    __shared__ float sc[kAttnRows][CAP];
    __shared__ float red[TPB][kAttnRows * LPT + 1][4];
    const uint32_t tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
    const uint32_t split = blockIdx.x, b = blockIdx.y;
    const uint32_t t0 = split * g.chunk, t1 = min(g.T, t0 + g.chunk);
    // operand offsets of this batch entry
    int64_t oq, ok, ov;
    uint32_t row0; // first row of this group in the program's [rows, T] space
    entry_offsets(g, b, oq, ok, ov, row0);
    const uint32_t l = tid % LPT, sub = tid / LPT;

    float4v kf[kAttnPasses], vf[kAttnPasses];
#pragma unroll
    for (int ps = 0; ps < kAttnPasses; ps++) {
        const uint32_t t = t0 + sub + ps * TPB;
        kf[ps] = (float4v){0.f, 0.f, 0.f, 0.f};
        vf[ps] = (float4v){0.f, 0.f, 0.f, 0.f};
        if (t < t1) {
            kf[ps] = *reinterpret_cast<const float4v *>(g.Kc + ok + (int64_t)t * g.k_st + l * 4);
            vf[ps] = *reinterpret_cast<const float4v *>(g.V + ov + (int64_t)t * g.v_st + l * 4);
        }
    }

    // ---- scores of the chunk: LPT lanes per position, one 16-byte piece of head_dim each
    {
        float4v qf[kAttnRows];
#pragma unroll
        for (int m = 0; m < kAttnRows; m++) {
            qf[m] = (float4v){0.f, 0.f, 0.f, 0.f};
            if ((uint32_t)m < g.M) qf[m] = *reinterpret_cast<const float4v *>(g.Q + oq + (int64_t)m * g.q_sm + l * 4);
        }
        const uint32_t passes = (t1 - t0 + TPB - 1) / TPB;
#pragma unroll
        for (int ps = 0; ps < kAttnPasses; ps++) {
            if ((uint32_t)ps < passes) {
                const uint32_t t = t0 + sub + ps * TPB;
#pragma unroll
                for (int m = 0; m < kAttnRows; m++) {
                    if ((uint32_t)m < g.M) {
                        float v = fmaf(qf[m][3], kf[ps][3], fmaf(qf[m][2], kf[ps][2], fmaf(qf[m][1], kf[ps][1], qf[m][0] * kf[ps][0])));
                        v = row16_sum(v);
                        if (LPT == 32) v = asf(fold_rows(asu(v), AddWords{}));
                        if (l == 0 && t < t1) sc[m][t - t0] = v;
                    }
                }
            }
        }
    }
    __syncthreads();

    // ---- the soft-max program on the chunk: a wave per query row, IPL positions per lane
    for (uint32_t m = wave; m < g.M; m += kBlock / 64) {
        const uint32_t row = row0 + m;
        int64_t base[P::nleaf + 1];
#pragma unroll
        for (int i = 0; i <= P::nleaf; i++) base[i] = 0;
        {
            uint32_t rr = row;
#pragma unroll
            for (uint32_t d = 0; d < (uint32_t)kMaxOuter; d++) {
                if (d >= a.g.nouter) break;
                const uint32_t q = fastdiv(rr, a.g.odiv[d]);
                const int64_t i = (int64_t)(rr - q * a.g.od[d]);
                rr = q;
#pragma unroll
                for (int lf = 1; lf < P::nleaf; lf++) base[lf] += i * a.leaf[lf].os[d];
            }
        }
        LeafWords<P, 1> w[IPL];
#pragma unroll
        for (int c = 0; c < IPL; c++) {
            const uint32_t i = lane + c * 64;
            if (i < t1 - t0) {
                aot_fetch_from<P, 1>(a, base, t0 + i, w[c]); // leaf 0 is the score
                w[c].v[0][0] = asu(sc[m][i]);
            }
        }
        uint32_t rs[kMaxRowReduce] = {0, 0, 0};
        uint32_t acc = row_init(true, true);
#pragma unroll
        for (int c = 0; c < IPL; c++) {
            if (lane + c * 64 < t1 - t0) {
                const Values<P, 1> s = aot_eval<P, 1, ri0>(w[c], rs, a.fault);
                acc = row_merge(true, true, acc, s.v[src0][0]);
            }
        }
        acc = wave_fold<1>(acc, [](uint32_t x, uint32_t y) { return row_merge(true, true, x, y); });
        rs[0] = acc;
        uint32_t sum = row_init(false, true);
#pragma unroll
        for (int c = 0; c < IPL; c++) {
            const uint32_t i = lane + c * 64;
            if (i < t1 - t0) {
                const Values<P, 1> s = aot_eval<P, 1, ri1>(w[c], rs, a.fault);
                sum = row_merge(false, true, sum, s.v[src1][0]);
                sc[m][i] = asf(s.v[src1][0]); // the un-normalised weight
            }
        }
        sum = wave_fold<1>(sum, [](uint32_t x, uint32_t y) { return row_merge(false, true, x, y); });
        if (lane == 0) {
            float *ml = g.part_ml + (((uint64_t)b * g.splits + split) * g.M + m) * 2;
            ml[0] = asf(acc);
            ml[1] = asf(sum);
        }
    }
    __syncthreads();

    // ---- weights times V: the lane's V pieces are those of its positions, head_dim piece l
    {
        float4v o[kAttnRows];
#pragma unroll
        for (int m = 0; m < kAttnRows; m++) o[m] = (float4v){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ps = 0; ps < kAttnPasses; ps++) {
            const uint32_t t = t0 + sub + ps * TPB;
            if (t < t1) {
#pragma unroll
                for (int m = 0; m < kAttnRows; m++) {
                    if ((uint32_t)m < g.M) {
                        const float wgt = sc[m][t - t0];
                        o[m][0] = fmaf(wgt, vf[ps][0], o[m][0]);
                        o[m][1] = fmaf(wgt, vf[ps][1], o[m][1]);
                        o[m][2] = fmaf(wgt, vf[ps][2], o[m][2]);
                        o[m][3] = fmaf(wgt, vf[ps][3], o[m][3]);
                    }
                }
            }
        }
#pragma unroll
        for (int m = 0; m < kAttnRows; m++)
            if ((uint32_t)m < g.M) {
#pragma unroll
                for (int j = 0; j < 4; j++) red[sub][m * LPT + l][j] = o[m][j];
            }
        __syncthreads();
        for (uint32_t e = tid; e < g.M * HD; e += kBlock) {
            const uint32_t m = e / HD, n = e % HD;
            float v = 0.0f;
#pragma unroll
            for (int k = 0; k < TPB; k++) v += red[k][m * LPT + n / 4][n % 4];
            g.part_o[(((uint64_t)b * g.splits + split) * g.M + m) * HD + n] = v;
        }
    }
}

// The same attention with ONE workgroup of 1024 threads per query row (and per half of head_dim, see VS) walking all
// T cached positions: no chunk results, no second launch.  At decode time a KV head's cache is a few hundred KiB to
// a few MiB, and the chunked pair of kernels spends most of its 20 us waiting (launch, operand offsets, a trip to
// memory, the hand-over to the combine, its trip).  Here the loads of K are asked for as far ahead as registers
// allow, the scores of the row wait in LDS, the soft-max program runs once over all of them (the row's maximum and
// sum cross the waves through LDS), V is on its way while that happens, and the weighted sum is divided by the
// row's sum where it is stored.  The workgroups of a batch entry (its query rows read the same K and V) get block
// indices a multiple of eight apart, which lands them on the same XCD: the second to last read hit in its L2.
// What bounds a workgroup is its compute unit's path to L2: measured, a compute unit streams about 60 GB/s (25 bytes a
// clock) out of L2 however many loads it keeps in flight (a ring of 16 passes per lane instead of two alternating trips
// of six was no faster), and a workgroup pulls all of K plus its half of V through it (835 KB at T = 2176: 14 us).
// Taken up to T = 4096 in one launch and, in
// two segments per row whose results decode_attention_combine_kernel merges, up to 8192; longer caches go to the chunked
// kernels, which spread a KV head over many workgroups.
// PASSES x (1024 / LPT) positions per trip to memory.  LOOP: several trips, the next always asked for before the
// current one is used (PASSES registers twice); else one trip covers T, the soft-max program's other leaves are
// asked for right behind K, and with at most ten passes V behind them (the registers hold both).
// VS = 2: the workgroup computes all scores but only one half of head_dim of the output, so that twice as many compute
// units pull on V (used when the launch would otherwise leave half of them idle).
constexpr int kRowBlock = 1024;
constexpr int kRowMaxT = 4096;
template <class P, int LPT, int PASSES, bool LOOP, int VS, class Heads>
__global__ __launch_bounds__(kRowBlock) void decode_attention_row_kernel(const AttnArgs g, const FusedArgs a, uint32_t *out, const Heads heads) {
    constexpr int HD = LPT * 4;
    constexpr bool RAW = std::is_same<Heads, RawHeads>::value;
    constexpr int TPB = kRowBlock / LPT; // positions per pass
    constexpr int SPAN = TPB * PASSES;    // positions per trip to memory
    constexpr int LPV = LPT / VS;         // lanes per position in the V phase
    constexpr int TPV = kRowBlock / LPV, PASSES_V = (PASSES + VS - 1) / VS, SPAN_V = TPV * PASSES_V;
    constexpr int WAVES = kRowBlock / 64;
    constexpr int IPL = LOOP ? kRowMaxT / kRowBlock : 1; // positions per thread in the soft-max phase
    constexpr bool V_EARLY = !LOOP && PASSES + PASSES_V <= 20;
    constexpr int ri0 = reduce_index<P>(0), ri1 = reduce_index<P>(1);
    constexpr int src0 = P::code[ri0][1], src1 = P::code[ri1][1];
    static_assert((P::code[ri0][0] & ~kInstrU32) == kRowMax && (P::code[ri1][0] & ~kInstrU32) == kRowSum,
                  "a soft-max: row maximum, then row sum");
    static_assert(LOOP || SPAN <= kRowBlock, "one position per thread in the soft-max phase");
    __shared__ float sc[LOOP ? kRowMaxT : kRowBlock];
    __shared__ float red[WAVES][HD / VS];
    __shared__ uint32_t cross[2][WAVES];
    const uint32_t tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
    // a cache beyond kRowMaxT positions is cut into segments over grid.y: a workgroup then leaves its segment's maximum,
    // sum and un-normalised weighted sum for decode_attention_combine_kernel
    const uint32_t seg = blockIdx.y, t_first = seg * g.chunk;
    const uint32_t T = min(g.T, t_first + g.chunk) - t_first; // positions of this workgroup
    // block -> (batch entry, query row, half): the workgroups of an entry eight blocks apart
    const uint32_t rest = blockIdx.x / 8, eight = fastdiv(rest, g.groups), inner = rest - eight * g.M * VS, m = inner / VS, part = inner % VS;
    const uint32_t b = eight * 8 + blockIdx.x % 8;
    if (b >= g.splits) return; // (the number of batch entries; the same for the whole workgroup)
    int64_t oq, ok, ov;
    uint32_t row0; // first row of this group in the program's [rows, T] space
    entry_offsets(g, b, oq, ok, ov, row0);
    const uint32_t l = tid % LPT, sub = tid / LPT, lv = tid % LPV, subv = tid / LPV;
    const uint32_t *kbase = g.Kc + ok + (int64_t)t_first * g.k_st + l * 4;
    const uint32_t *vbase = g.V + ov + (int64_t)t_first * g.v_st + (part * LPV + lv) * 4;
    // the trip that starts at `first`.  Positions beyond the last are clamped, not tested: with a test in front of every load the
    // compiler knows of none that is on its way, and the first score waits for all of K and V.  (What they bring is not used.)
    auto ask_k_at = [&](float4v (&f)[PASSES], uint32_t first) {
#pragma unroll
        for (int ps = 0; ps < PASSES; ps++) f[ps] = *reinterpret_cast<const float4v *>(kbase + (int64_t)min(first + sub + ps * TPB, T - 1) * g.k_st);
    };
    auto ask_v_at = [&](float4v (&f)[PASSES_V], uint32_t first) {
#pragma unroll
        for (int ps = 0; ps < PASSES_V; ps++) f[ps] = *reinterpret_cast<const float4v *>(vbase + (int64_t)min(first + subv + ps * TPV, T - 1) * g.v_st);
    };
    // (tag types: a trip inside the T positions, and one that ends beyond them)
    constexpr std::true_type whole_trip{};
    constexpr std::false_type ragged{};
    float4v ka[PASSES], kb[LOOP ? PASSES : 1];
    float4v va[PASSES_V], vb[LOOP ? PASSES_V : 1];
    // (loads come back in the order in which they are asked for: the query and K, the leaves, V)
    float4v qf;
    const bool last = RAW && t_first + T == g.T; // this workgroup's positions end with the newest row
    const uint32_t cached = T - last;
    const uint32_t uwave = __builtin_amdgcn_readfirstlane(wave);
    OpenHead<LPT> mine; // the first wave finishes q, the second the newest row
    if constexpr (RAW) {
        const uint32_t seq = fastdiv(b, heads.heads), head = b - seq * heads.heads.d;
        if (uwave == 0) mine.load(heads.q, (uint64_t)seq * heads.q.n + (head * g.M + m) * HD, l);
        else if (uwave == 1) mine.load(heads.k, (uint64_t)seq * heads.k.n + head * HD, l);
    } else {
        qf = *reinterpret_cast<const float4v *>(g.Q + oq + (int64_t)m * g.q_sm + l * 4);
    }
    ask_k_at(ka, 0);
    // the soft-max program's other leaves at this thread's positions (tid, tid + 1024, ...)
    LeafWords<P, 1> w[IPL];
    int64_t base[P::nleaf + 1];
    leaf_offsets<P>(a, row0 + m, base);
    auto fetch_leaves = [&]() {
#pragma unroll
        for (int c = 0; c < IPL; c++)
            aot_fetch_from<P, 1>(a, base, t_first + min(tid + c * kRowBlock, T - 1), w[c]);
    };
    if constexpr (!LOOP) fetch_leaves(); // nothing waits for them yet
    if constexpr (V_EARLY) ask_v_at(va, 0);

    // ---- scores of the whole row
    auto score_of = [&](const float4v &k) {
        float v = fmaf(qf[3], k[3], fmaf(qf[2], k[2], fmaf(qf[1], k[1], qf[0] * k[0])));
        v = row16_sum(v);
        if (LPT == 32) v = asf(fold_rows(asu(v), AddWords{}));
        return v;
    };
    if constexpr (RAW) {
        float *const rows = &red[0][0]; // q, the newest row (red itself is needed behind the soft-max)
        if (uwave < 2) {
            const float4v v = mine.finish(uwave == 0 ? heads.q : heads.k, l);
            if (lane < LPT) {
                *reinterpret_cast<float4v *>(rows + uwave * HD + l * 4) = v;
                uint32_t *const to = const_cast<uint32_t *>(uwave == 0 ? g.Q + oq + (int64_t)m * g.q_sm : g.Kc + ok + (int64_t)(g.T - 1) * g.k_st);
                if (part == 0 && (uwave == 0 ? seg == 0 : last && m == 0)) *reinterpret_cast<float4v *>(to + l * 4) = v;
            }
        }
        __syncthreads();
        qf = *reinterpret_cast<const float4v *>(rows + l * 4);
        if (last && uwave == 0) {
            const float v = score_of(*reinterpret_cast<const float4v *>(rows + HD + l * 4));
            if (lane == 0) sc[cached] = v;
        }
    }
    auto score = [&](const float4v (&f)[PASSES], uint32_t first, auto full) {
#pragma unroll
        for (int ps = 0; ps < PASSES; ps++) {
            const uint32_t t = first + sub + ps * TPB;
            if (decltype(full)::value || first + ps * TPB < cached) { // the same for the whole workgroup
                const float v = score_of(f[ps]);
                if (l == 0 && (decltype(full)::value || t < cached)) sc[t] = v;
            }
        }
    };
    auto score_at = [&](const float4v (&f)[PASSES], uint32_t first) {
        if (first + SPAN <= cached) score(f, first, whole_trip);
        else score(f, first, ragged);
    };
    if constexpr (LOOP) {
        for (uint32_t first = 0; first < T; first += 2 * SPAN) {
            if (first + SPAN < T) ask_k_at(kb, first + SPAN);
            score_at(ka, first);
            if (first + 2 * SPAN < T) ask_k_at(ka, first + 2 * SPAN);
            if (first + SPAN < T) score_at(kb, first + SPAN);
        }
    } else {
        score_at(ka, 0);
    }
    if constexpr (!V_EARLY) ask_v_at(va, 0); // on its way through the soft-max
    if constexpr (LOOP) fetch_leaves();
    __syncthreads();

    // ---- the soft-max program over the row
    float total, row_max;
    {
        uint32_t rs[kMaxRowReduce] = {0, 0, 0};
        uint32_t acc = row_init(true, true);
#pragma unroll
        for (int c = 0; c < IPL; c++) {
            const uint32_t i = tid + c * kRowBlock;
            if (i < T) {
                w[c].v[0][0] = asu(sc[i]); // leaf 0 is the score
                const Values<P, 1> s = aot_eval<P, 1, ri0>(w[c], rs, a.fault);
                acc = row_merge(true, true, acc, s.v[src0][0]);
            }
        }
        acc = wave_fold<1>(acc, [](uint32_t x, uint32_t y) { return row_merge(true, true, x, y); });
        if (lane == 0) cross[0][wave] = acc;
        __syncthreads();
        acc = cross[0][0];
#pragma unroll
        for (int k = 1; k < WAVES; k++) acc = row_merge(true, true, acc, cross[0][k]);
        rs[0] = acc;
        row_max = asf(acc);
        uint32_t sum = row_init(false, true);
#pragma unroll
        for (int c = 0; c < IPL; c++) {
            const uint32_t i = tid + c * kRowBlock;
            if (i < T) {
                const Values<P, 1> s = aot_eval<P, 1, ri1>(w[c], rs, a.fault);
                sum = row_merge(false, true, sum, s.v[src1][0]);
                sc[i] = asf(s.v[src1][0]); // the un-normalised weight
            }
        }
        sum = wave_fold<1>(sum, [](uint32_t x, uint32_t y) { return row_merge(false, true, x, y); });
        if (lane == 0) cross[1][wave] = sum;
        __syncthreads();
        sum = cross[1][0];
#pragma unroll
        for (int k = 1; k < WAVES; k++) sum = row_merge(false, true, sum, cross[1][k]);
        total = asf(sum);
    }

    // ---- weights times V (this workgroup's columns)
    float4v o = {0.f, 0.f, 0.f, 0.f};
    auto weigh = [&](const float4v (&f)[PASSES_V], uint32_t first, auto full) {
#pragma unroll
        for (int ps = 0; ps < PASSES_V; ps++) {
            const uint32_t t = first + subv + ps * TPV;
            if (decltype(full)::value || t < T) {
                const float wgt = sc[t];
                o[0] = fmaf(wgt, f[ps][0], o[0]);
                o[1] = fmaf(wgt, f[ps][1], o[1]);
                o[2] = fmaf(wgt, f[ps][2], o[2]);
                o[3] = fmaf(wgt, f[ps][3], o[3]);
            }
        }
    };
    auto weigh_at = [&](const float4v (&f)[PASSES_V], uint32_t first) {
        if (first + SPAN_V <= T) weigh(f, first, whole_trip);
        else weigh(f, first, ragged);
    };
    if constexpr (LOOP) {
        for (uint32_t first = 0; first < T; first += 2 * SPAN_V) {
            if (first + SPAN_V < T) ask_v_at(vb, first + SPAN_V);
            weigh_at(va, first);
            if (first + 2 * SPAN_V < T) ask_v_at(va, first + 2 * SPAN_V);
            if (first + SPAN_V < T) weigh_at(vb, first + SPAN_V);
        }
    } else {
        weigh_at(va, 0);
    }
    // the wave's position groups (lanes lv, lv + LPV, ...) first, then the waves through LDS
#pragma unroll
    for (int j = 0; j < 4; j++) o[j] = wave_add_up<LPV>(o[j]);
    if (lane < LPV) *reinterpret_cast<float4v *>(&red[wave][lv * 4]) = o;
    __syncthreads();
    if (tid < HD / VS) {
        float v = 0.0f;
#pragma unroll
        for (int k = 0; k < WAVES; k++) v += red[k][tid];
        if (g.part_o) {
            const uint64_t at = ((uint64_t)b * gridDim.y + seg) * g.M + m;
            g.part_o[at * HD + part * (HD / VS) + tid] = v;
            if (tid == 0 && part == 0) {
                g.part_ml[at * 2] = row_max;
                g.part_ml[at * 2 + 1] = total;
            }
        } else {
            out[((uint64_t)b * g.M + m) * HD + part * (HD / VS) + tid] = asu(v / total);
        }
    }
}

// The same attention with a workgroup of 1024 threads per (batch entry, KV head) x SEGMENT of the cached positions,
// all of the group's query rows together: every byte of K and V crosses the path from L2 into a compute unit once
// (one workgroup per query row pulls K through it once per row and per half of head_dim: six times the traffic, and
// that path, 25 bytes a clock per unit, is what bounds a launch of this size).  With 256 / (batch entries x KV heads)
// segments a launch puts one workgroup on every compute unit, each with T / segments positions: 134 KB of K and V at
// the 1B shape's T = 2100, in flight at once (PASSES x 1024 / LPT positions per trip, K and V of a trip in 2 x PASSES
// sixteen-byte loads per lane).  A segment leaves its rows' maximum, sum and un-normalised weighted sum of V, as the
// chunked kernel does; decode_attention_combine_kernel merges the segments.
// LOOP: several trips, the next always asked for before the current one is used; else one trip covers the segment and
// the soft-max program's other leaves are asked for between K and V.  MM: most query rows per KV head (4 or 8).
constexpr int kSegBlock = 1024;
constexpr int kSegMaxChunk = 2048; // most positions per workgroup: their scores wait in LDS, MM x 8 KiB
constexpr size_t seg_lds_bytes(int mm, int hd, uint32_t chunk) {
    return ((size_t)mm * ((chunk + 63) / 64 * 64) + (size_t)(kSegBlock / 64) * mm * hd) * sizeof(float);
}
template <class P, int LPT, int MM, int PASSES, bool LOOP, class Heads>
__global__ __launch_bounds__(kSegBlock) void decode_attention_seg_kernel(const AttnArgs g, const FusedArgs a, const Heads heads) {
    constexpr int HD = LPT * 4;
    constexpr bool RAW = std::is_same<Heads, RawHeads>::value;
    constexpr int TPB = kSegBlock / LPT; // positions per pass
    constexpr int SPAN = TPB * PASSES;    // positions per trip to memory
    constexpr int WAVES = kSegBlock / 64;
    constexpr int IPL = LOOP ? 1 : (SPAN + 63) / 64; // positions per lane in the soft-max phase whose leaves wait in registers
    constexpr int ri0 = reduce_index<P>(0), ri1 = reduce_index<P>(1);
    constexpr int src0 = P::code[ri0][1], src1 = P::code[ri1][1];
    static_assert((P::code[ri0][0] & ~kInstrU32) == kRowMax && (P::code[ri1][0] & ~kInstrU32) == kRowSum,
                  "a soft-max: row maximum, then row sum");
    extern __shared__ float seg_lds[];
    const uint32_t cap = (g.chunk + 63) / 64 * 64;
    float *sc = seg_lds;              // [MM][cap]: scores, then un-normalised weights
    float *red = seg_lds + MM * cap;  // [WAVES][MM * HD]
    const uint32_t tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
    const uint32_t split = blockIdx.x, b = blockIdx.y;
    const uint32_t t0 = split * g.chunk, n = min(g.T, t0 + g.chunk) - t0; // (the host makes no empty segment)
    int64_t oq, ok, ov;
    uint32_t row0; // first row of this group in the program's [rows, T] space
    entry_offsets(g, b, oq, ok, ov, row0);
    const uint32_t l = tid % LPT, sub = tid / LPT;
    const uint32_t *kbase = g.Kc + ok + (int64_t)t0 * g.k_st + l * 4;
    const uint32_t *vbase = g.V + ov + (int64_t)t0 * g.v_st + l * 4;
    // the trip that starts at `first` (positions clamped as in the kernel above)
    auto ask = [&](float4v (&f)[PASSES], const uint32_t *base, int64_t st, uint32_t first) {
#pragma unroll
        for (int ps = 0; ps < PASSES; ps++) f[ps] = *reinterpret_cast<const float4v *>(base + (int64_t)min(first + sub + ps * TPB, n - 1) * st);
    };
    constexpr std::true_type whole_trip{};
    constexpr std::false_type ragged{};
    auto ask_k = [&](float4v (&f)[PASSES], uint32_t first) { ask(f, kbase, g.k_st, first); };
    auto ask_v = [&](float4v (&f)[PASSES], uint32_t first) { ask(f, vbase, g.v_st, first); };
    float4v ka[PASSES], kb[LOOP ? PASSES : 1];
    float4v va[PASSES], vb[LOOP ? PASSES : 1];
    float4v qf[MM];
    const bool last = RAW && split + 1 == g.splits; // this segment ends with the newest row
    const uint32_t cached = n - last;
    const uint32_t uwave = __builtin_amdgcn_readfirstlane(wave);
    OpenHead<LPT> mine; // a wave finishes a row of q each, the next one the newest row of K
    if constexpr (RAW) {
        const uint32_t seq = fastdiv(b, heads.heads), head = b - seq * heads.heads.d;
        if (uwave < g.M) mine.load(heads.q, (uint64_t)seq * heads.q.n + (head * g.M + uwave) * HD, l);
        else if (uwave == g.M) mine.load(heads.k, (uint64_t)seq * heads.k.n + head * HD, l);
    } else {
#pragma unroll
        for (int m = 0; m < MM; m++) {
            qf[m] = *reinterpret_cast<const float4v *>(g.Q + oq + (int64_t)min((uint32_t)m, g.M - 1) * g.q_sm + l * 4);
        }
    }
    ask_k(ka, 0);
    // the soft-max phase gives a wave a query row (waves M.. have none); its lanes take positions lane, lane + 64, ...
    const uint32_t my_row = wave; // < g.M: this wave runs the program on row my_row
    int64_t base[P::nleaf + 1];
    LeafWords<P, 1> w[IPL];
    leaf_offsets<P>(a, row0 + min(my_row, g.M - 1), base);
    if constexpr (!LOOP) { // nothing waits for them yet
#pragma unroll
        for (int c = 0; c < IPL; c++) aot_fetch_from<P, 1>(a, base, t0 + min(lane + c * 64, n - 1), w[c]);
        ask_v(va, 0); // the whole segment is in flight: the registers hold both
    }


    // ---- scores of the segment, all rows of the group
    auto score_of = [&](int m, const float4v &k) {
        float v = fmaf(qf[m][3], k[3], fmaf(qf[m][2], k[2], fmaf(qf[m][1], k[1], qf[m][0] * k[0])));
        v = row16_sum(v);
        if (LPT == 32) v = asf(fold_rows(asu(v), AddWords{}));
        return v;
    };
    if constexpr (RAW) {
        static_assert(MM < WAVES, "a wave per row");
        // (red is needed behind the soft-max: until then it holds the finished rows, K's behind q's)
        if (uwave <= g.M) {
            const float4v v = mine.finish(uwave < g.M ? heads.q : heads.k, l);
            if (lane < LPT) {
                *reinterpret_cast<float4v *>(red + uwave * HD + l * 4) = v;
                uint32_t *const to = const_cast<uint32_t *>(uwave < g.M ? g.Q + oq + (int64_t)uwave * g.q_sm : g.Kc + ok + (int64_t)(g.T - 1) * g.k_st);
                if (uwave < g.M ? split == 0 : last) *reinterpret_cast<float4v *>(to + l * 4) = v;
            }
        }
        __syncthreads();
#pragma unroll
        for (int m = 0; m < MM; m++) qf[m] = *reinterpret_cast<const float4v *>(red + min((uint32_t)m, g.M - 1) * HD + l * 4);
        if (last && uwave == 0) {
            const float4v newest = *reinterpret_cast<const float4v *>(red + g.M * HD + l * 4);
#pragma unroll
            for (int m = 0; m < MM; m++) {
                if ((uint32_t)m < g.M) {
                    const float v = score_of(m, newest);
                    if (lane == 0) sc[m * cap + cached] = v;
                }
            }
        }
    }
    auto score = [&](const float4v (&f)[PASSES], uint32_t first, auto full) {
#pragma unroll
        for (int ps = 0; ps < PASSES; ps++) {
            const uint32_t t = first + sub + ps * TPB;
            if (decltype(full)::value || first + ps * TPB < cached) { // the same for the whole workgroup
#pragma unroll
                for (int m = 0; m < MM; m++) {
                    if ((uint32_t)m < g.M) {
                        const float v = score_of(m, f[ps]);
                        if (l == 0 && (decltype(full)::value || t < cached)) sc[m * cap + t] = v;
                    }
                }
            }
        }
    };
    auto score_at = [&](const float4v (&f)[PASSES], uint32_t first) {
        if (first + SPAN <= cached) score(f, first, whole_trip);
        else score(f, first, ragged);
    };
    if constexpr (LOOP) {
        for (uint32_t first = 0; first < n; first += 2 * SPAN) {
            if (first + SPAN < n) ask_k(kb, first + SPAN);
            score_at(ka, first);
            if (first + 2 * SPAN < n) ask_k(ka, first + 2 * SPAN);
            if (first + SPAN < n) score_at(kb, first + SPAN);
        }
    } else {
        score_at(ka, 0);
    }
    if constexpr (LOOP) ask_v(va, 0); // on its way through the soft-max
    __syncthreads();

    // ---- the soft-max program on the segment: local maximum, local sum, un-normalised weights
    if (my_row < g.M) {
        const uint32_t m = my_row;
        uint32_t rs[kMaxRowReduce] = {0, 0, 0};
        uint32_t acc = row_init(true, true);
        if constexpr (!LOOP) {
#pragma unroll
            for (int c = 0; c < IPL; c++) {
                const uint32_t i = lane + c * 64;
                if (i < n) {
                    w[c].v[0][0] = asu(sc[m * cap + i]); // leaf 0 is the score
                    const Values<P, 1> s = aot_eval<P, 1, ri0>(w[c], rs, a.fault);
                    acc = row_merge(true, true, acc, s.v[src0][0]);
                }
            }
        } else {
            for (uint32_t i = lane; i < n; i += 64) {
                aot_fetch_from<P, 1>(a, base, t0 + i, w[0]);
                w[0].v[0][0] = asu(sc[m * cap + i]);
                const Values<P, 1> s = aot_eval<P, 1, ri0>(w[0], rs, a.fault);
                acc = row_merge(true, true, acc, s.v[src0][0]);
            }
        }
        acc = wave_fold<1>(acc, [](uint32_t x, uint32_t y) { return row_merge(true, true, x, y); });
        rs[0] = acc;
        uint32_t sum = row_init(false, true);
        if constexpr (!LOOP) {
#pragma unroll
            for (int c = 0; c < IPL; c++) {
                const uint32_t i = lane + c * 64;
                if (i < n) {
                    const Values<P, 1> s = aot_eval<P, 1, ri1>(w[c], rs, a.fault);
                    sum = row_merge(false, true, sum, s.v[src1][0]);
                    sc[m * cap + i] = asf(s.v[src1][0]); // the un-normalised weight
                }
            }
        } else {
            for (uint32_t i = lane; i < n; i += 64) {
                aot_fetch_from<P, 1>(a, base, t0 + i, w[0]);
                w[0].v[0][0] = asu(sc[m * cap + i]);
                const Values<P, 1> s = aot_eval<P, 1, ri1>(w[0], rs, a.fault);
                sum = row_merge(false, true, sum, s.v[src1][0]);
                sc[m * cap + i] = asf(s.v[src1][0]);
            }
        }
        sum = wave_fold<1>(sum, [](uint32_t x, uint32_t y) { return row_merge(false, true, x, y); });
        if (lane == 0) {
            float *ml = g.part_ml + (((uint64_t)b * g.splits + split) * g.M + m) * 2;
            ml[0] = asf(acc);
            ml[1] = asf(sum);
        }
    }
    __syncthreads();

    // ---- weights times V: the lane's pieces of V are those of its positions, piece l of head_dim
    float4v o[MM];
#pragma unroll
    for (int m = 0; m < MM; m++) o[m] = (float4v){0.f, 0.f, 0.f, 0.f};
    auto weigh = [&](const float4v (&f)[PASSES], uint32_t first, auto full) {
#pragma unroll
        for (int ps = 0; ps < PASSES; ps++) {
            const uint32_t t = first + sub + ps * TPB;
            if (decltype(full)::value || t < n) {
#pragma unroll
                for (int m = 0; m < MM; m++) {
                    if ((uint32_t)m < g.M) {
                        const float wgt = sc[m * cap + t];
                        o[m][0] = fmaf(wgt, f[ps][0], o[m][0]);
                        o[m][1] = fmaf(wgt, f[ps][1], o[m][1]);
                        o[m][2] = fmaf(wgt, f[ps][2], o[m][2]);
                        o[m][3] = fmaf(wgt, f[ps][3], o[m][3]);
                    }
                }
            }
        }
    };
    auto weigh_at = [&](const float4v (&f)[PASSES], uint32_t first) {
        if (first + SPAN <= n) weigh(f, first, whole_trip);
        else weigh(f, first, ragged);
    };
    if constexpr (LOOP) {
        for (uint32_t first = 0; first < n; first += 2 * SPAN) {
            if (first + SPAN < n) ask_v(vb, first + SPAN);
            weigh_at(va, first);
            if (first + 2 * SPAN < n) ask_v(va, first + 2 * SPAN);
            if (first + SPAN < n) weigh_at(vb, first + SPAN);
        }
    } else {
        weigh_at(va, 0);
    }
    // the wave's position groups (lanes l, l + LPT, ...) first, then the waves through LDS
#pragma unroll
    for (int m = 0; m < MM; m++) {
        if ((uint32_t)m < g.M) {
#pragma unroll
            for (int j = 0; j < 4; j++) o[m][j] = wave_add_up<LPT>(o[m][j]);
            if (lane < LPT) *reinterpret_cast<float4v *>(&red[(wave * MM + m) * HD + l * 4]) = o[m];
        }
    }
    __syncthreads();
    for (uint32_t e = tid; e < g.M * HD; e += kSegBlock) {
        const uint32_t m = e / HD, d = e % HD;
        float v = 0.0f;
#pragma unroll
        for (int k = 0; k < WAVES; k++) v += red[(k * MM + m) * HD + d];
        g.part_o[(((uint64_t)b * g.splits + split) * g.M + m) * HD + d] = v;
    }
}

// out[b][m][n] = sum_c e^(m_c - g) o_c[n] / sum_c e^(m_c - g) l_c.  A workgroup per (batch entry, query row), whose waves share the
// chunks: lane c first holds the statistics of chunk c (each wave computes each weight e^(m_c - g) once and reads it from that lane), then
// lane n sums output element n (and n + 64) over the wave's chunks, and the waves' sums meet in LDS.
// Bound by latency: one trip to memory.  A wave per row, with a shuffle per chunk, took 4.74 us for 16 rows of 32 chunks of 128; so 2.83 (3.33 in
// Qwen3-0.6B's steps, behind the segments).
__global__ __launch_bounds__(kBlock) void decode_attention_combine_kernel(const float *part_o, const float *part_ml, uint32_t *out, uint32_t splits, uint32_t M, uint32_t hd) {
    constexpr uint32_t kWaves = kBlock / 64, kTrip = 64, kMine = kTrip / kWaves; // chunks per trip, of which a wave takes every fourth
    __shared__ float sums[kWaves][2][64];
    const uint32_t lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const uint64_t r = blockIdx.x, b = r / M;
    const uint32_t m = (uint32_t)(r - b * M);
    const float *ml = part_ml + (b * splits * M + m) * 2; // chunk c at + c * M * 2
    const float *po = part_o + (b * splits * M + m) * (uint64_t)hd; // chunk c at + c * M * hd
    const uint32_t d0 = min(lane, hd - 1), d1 = min(lane + 64, hd - 1);
    float gmax = kF32Min, num0 = 0.0f, num1 = 0.0f, den = 0.0f;
    for (uint32_t c0 = 0; c0 < splits; c0 += kTrip) {
        // every load of the trip is asked for before anything is used (a chunk behind the last: the last one's, taken as zero)
        const uint32_t c = min(c0 + lane, splits - 1);
        const float2 mine = *reinterpret_cast<const float2 *>(ml + (uint64_t)c * M * 2);
        float v0[kMine], v1[kMine];
#pragma unroll
        for (uint32_t k = 0; k < kMine; k++) {
            const float *o = po + (uint64_t)min(c0 + wave + k * kWaves, splits - 1) * M * hd;
            v0[k] = o[d0];
            v1[k] = o[d1];
        }
        const bool there = c0 + lane < splits;
        const float m2 = fmaxf(gmax, asf(wave_fold<1>(asu(there ? mine.x : kF32Min), LargerWords{})));
        // what was summed so far is relative to the old maximum
        const float rescale = expf(gmax - m2), w = there ? expf(mine.x - m2) : 0.0f;
        gmax = m2;
        num0 *= rescale;
        num1 *= rescale;
        den = fmaf(w, there ? mine.y : 0.0f, den * rescale);
#pragma unroll
        for (uint32_t k = 0; k < kMine; k++) {
            const uint32_t at = wave + k * kWaves;
            const bool in = c0 + at < splits;
            const float wk = asf((uint32_t)__builtin_amdgcn_readlane((int)asu(w), (int)at));
            num0 = fmaf(wk, in ? v0[k] : 0.0f, num0);
            num1 = fmaf(wk, in ? v1[k] : 0.0f, num1);
        }
    }
    den = wave_add<1>(den); // (every wave has all chunks' sums)
    sums[wave][0][lane] = num0;
    sums[wave][1][lane] = num1;
    __syncthreads();
    const uint32_t d = threadIdx.x;
    if (d >= hd) return; // (hd <= 128: the first two waves)
    float s = 0.0f;
#pragma unroll
    for (uint32_t k = 0; k < kWaves; k++) s += sums[k][d / 64][d % 64];
    out[r * hd + d] = asu(s / den);
}

// ---- prefill: causal attention of many query rows in one pass ---------------------------------------------------
// The same three ops as above with thousands of query rows per KV head: unfused they write and re-read the
// [rows, T] score matrix four times (2 GiB per layer of the 1B-shape prefill).  Here a workgroup takes 128
// query rows of one KV head (a wave 32 of them) and walks the cached positions in tiles of 64, never going
// beyond the last position its rows may see.  Everything is computed TRANSPOSED, so that a query is a lane:
//     S^T[t][m] = K[t] . Q[m] / scale  first MFMA operand K (from LDS), second Q / scale (registers, loaded once)
//     running maximum / sum per query  = per lane: in-register over its 32 values + one exchange with lane ^ 32
//     O^T[d][m] += V^T[d][t] P^T[t][m] first operand V^T (columns of the LDS tile), second P^T — which, in the accumulator
//                                      layout of the 32x32 instructions (column = lane % 32, rows 8*(v/4) +
//                                      4*(lane/32) + v%4), already is the operand layout: no trip through LDS
// The scores are divided by the scale and masked exactly as the soft-max program does (x / d + f32(i < j) * m with
// i the query's position, j the key's); masked keys get weight zero, which is what exp(x - max) rounds to for them.
// out = O / l at the end (the program divides the weights first: same value up to rounding).
// Bound by the matrix pipes, and in pieces by them and the splitting together: 2 x 2 x 32 x 64 x 64 flop per wave and tile over
// ~half of the [rows, T] rectangle.
struct PrefillArgs {
    uint32_t *out;      // [batch][M][hd], dense
    uint32_t S;         // query positions per head: row m of a group is position m % S
    uint32_t pos0;      // position of the first query row (length of the cache before this chunk)
    uint32_t scale;     // f32 bits of the divisor of the scores
    uint32_t mask_mul;  // f32 bits of the multiplier of the 0/1 mask
    uint32_t batch;     // folded batch entries (KV heads)
    uint32_t tiles_per_head; // S / 128 when that is whole and heads are whole in M, else 0
    // Few workgroups (one sequence, a short prompt): the keys of a row tile are cut into `ksplit` parts over grid.y; a part
    // leaves its rows' running maximum, sum and un-normalised O for prefill_attention_combine_kernel.
    uint32_t ksplit;    // 1: none
    float *part_o;      // [ksplit][batch][M][hd]
    float *part_ml;     // [ksplit][batch][M][2]
};

constexpr int kPfRows = 128, kPfKeys = 64;
// The 32-bit instructions' K and V tiles, [64 keys][head_dim + 4] each (a row starts 4 banks after the one before), double
// buffered: 68 KiB for head_dim 64 (two workgroups per CU), 132 KiB for 128 (one).  The pieces take 48 KiB of it, one buffer:
// the next tile waits in registers (and at head_dim 64 the other workgroup covers the second barrier).
constexpr size_t prefill_lds_bytes(int hd) { return 2 * 2 * (size_t)kPfKeys * (hd + 4) * sizeof(float); }

// PIECES: both products as products of bfloat16 pieces (split_tile.hpp), 2.67 times the rate of the 32-bit instructions: the
// queries' pieces stay in registers, those of K and V are made on the way into LDS, once for the four waves (V turned, so that a
// fragment's eight keys are the eight that a lane holds weights of), and the weights are split in place.  Returns true, and has
// stored nothing, if a value lies at the ends of the range that pieces cover; !PIECES: the 32-bit instructions.
// Measured, 32-bit instructions -> pieces: 4 x 2048 tokens, 32 heads of 64 over 8 KV heads 626 -> 433 us (159 TFLOP/s of the visible
// half); 1024 tokens, 16 heads of 128 over 8 85 -> 78; 512 tokens, 9 heads of 64 over 3 19.6 -> 17.0; 4 x 8 tokens 12.7 -> 12.9.  The
// products are no longer what bounds it alone: splitting K, V and the weights, the exponentials and the two barriers of a tile weigh as
// much.  Error against 64 bits: 4.0e-7 -> 2.1e-7 (the first of these).  With a value beyond the range in every head both ways are run:
// the whole call of the first 666 -> 841 us (442 without such a value), of the second 95 -> 110.
template <int HD, bool PIECES> __device__ __forceinline__ bool prefill_rows(const AttnArgs &g, const PrefillArgs &e, float *const pf_lds) {
    static_assert(HD == 64 || HD == 128, "head_dim 64 or 128");
    constexpr int KEYS = PIECES && HD == 128 ? 32 : kPfKeys; // per tile
    constexpr int kPfPitch = HD + 4;
    typedef float float16v __attribute__((ext_vector_type(16)));
    float (*Ks)[kPfKeys][kPfPitch] = reinterpret_cast<float (*)[kPfKeys][kPfPitch]>(pf_lds);                       // [2][t][d]
    float (*Vs)[kPfKeys][kPfPitch] = reinterpret_cast<float (*)[kPfKeys][kPfPitch]>(pf_lds + 2 * kPfKeys * kPfPitch); // [2][t][d]
    const uint32_t tid = threadIdx.x, lane = tid % 64, wave = tid / 64, li = lane % 32, lg = lane / 32;
    // Work per workgroup grows with the position of its rows inside their head (more visible keys), so the grid
    // is walked longest first over ALL batch entries and heads: the tail of the launch is made of short ones.
    const uint32_t ntile_rows = (g.M + kPfRows - 1) / kPfRows;
    uint32_t rt, b;
    if (e.tiles_per_head) {
        const uint32_t per_step = e.batch * (ntile_rows / e.tiles_per_head); // workgroups with the same row position
        const uint32_t step = blockIdx.x / per_step, rest = blockIdx.x % per_step;
        rt = (rest / e.batch) * e.tiles_per_head + (e.tiles_per_head - 1 - step);
        b = rest % e.batch;
    } else { // heads are not whole numbers of row tiles
        rt = ntile_rows - 1 - blockIdx.x / e.batch;
        b = blockIdx.x % e.batch;
    }
    int64_t oq = 0, ok = 0, ov = 0;
    {
        uint32_t bb = b;
        for (uint32_t d = 0; d < g.nb; d++) {
            const uint32_t q = fastdiv(bb, g.bdiv[d]);
            const int64_t i = (int64_t)(bb - q * g.bd[d]);
            bb = q;
            oq += i * g.q_bs[d];
            ok += i * g.k_bs[d];
        }
        bb = b;
        for (uint32_t d = 0; d < g.nbv; d++) {
            const uint32_t q = fastdiv(bb, g.vbdiv[d]);
            const int64_t i = (int64_t)(bb - q * g.vbd[d]);
            bb = q;
            ov += i * g.v_bs[d];
        }
    }
    const uint32_t m0 = rt * kPfRows;
    const uint32_t m = m0 + wave * 32 + li; // this lane's query row (both halves of the wave hold the same 32 queries)
    const bool live = m < g.M;
    const uint32_t iq = e.pos0 + (live ? m % e.S : 0); // position of the query: keys up to iq are visible
    // last key any row of the workgroup may see
    uint32_t kmax;
    {
        const uint32_t s0 = m0 % e.S, last = min(m0 + kPfRows, g.M) - 1 - m0; // rows m0 .. m0 + last
        const uint32_t smax = s0 + last < e.S ? s0 + last : e.S - 1;            // the tile may run into the next head
        kmax = min(g.T - 1, e.pos0 + smax);
    }
    const uint32_t ntiles_all = kmax / kPfKeys + 1;
    // this workgroup's share of the key tiles (all of them without a split), the same for either way to multiply
    const uint32_t per_part = (ntiles_all + e.ksplit - 1) / e.ksplit;
    const uint32_t it_first = blockIdx.y * per_part * (kPfKeys / KEYS);
    const uint32_t ntiles = min(kmax / KEYS + 1, (blockIdx.y + 1) * per_part * (kPfKeys / KEYS));

    // the query rows, as second MFMA operands: chunk c covers d = 8c .. 8c+7, this lane holds 4*lg .. 4*lg+3 of them.
    // The program divides every score by the scale; dividing the query once instead is the same value up to
    // rounding and takes the division out of the loop.
    const float scale = asf(e.scale);
    typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
    typedef uint32_t uint4w __attribute__((ext_vector_type(4)));
    float4v qf[PIECES ? 1 : HD / 8];
    bf16x8 qp[PIECES ? HD / 16 : 1][3]; // chunk c: d = 16 c + 8 lg .. + 7
    float top_qk = 0.0f, top_v = 0.0f; // largest magnitudes seen
    if constexpr (!PIECES) {
#pragma unroll
        for (int c = 0; c < HD / 8; c++) {
            qf[c] = (float4v){0.f, 0.f, 0.f, 0.f};
            if (live) qf[c] = *reinterpret_cast<const float4v *>(g.Q + oq + (int64_t)m * g.q_sm + c * 8 + lg * 4);
#pragma unroll
            for (int r = 0; r < 4; r++) qf[c][r] = qf[c][r] / scale;
        }
    } else {
#pragma unroll
        for (int c = 0; c < HD / 16; c++) {
            uint4w w[3];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                float4v q = {0.f, 0.f, 0.f, 0.f};
                if (live) q = *reinterpret_cast<const float4v *>(g.Q + oq + (int64_t)m * g.q_sm + c * 16 + lg * 8 + h * 4);
#pragma unroll
                for (int r = 0; r < 4; r++) q[r] = q[r] / scale;
                split::grow(top_qk, q[0], q[1]);
                split::grow(top_qk, q[2], q[3]);
                uint32_t a[3], b[3];
                split::split2(q[0], q[1], a);
                split::split2(q[2], q[3], b);
#pragma unroll
                for (int p = 0; p < 3; p++) w[p][2 * h] = a[p], w[p][2 * h + 1] = b[p];
            }
#pragma unroll
            for (int p = 0; p < 3; p++) qp[c][p] = __builtin_bit_cast(bf16x8, w[p]);
        }
    }
    float16v acc_o[HD / 32];
#pragma unroll
    for (int db = 0; db < HD / 32; db++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc_o[db][v] = 0.0f;
    float run_max = -INFINITY, run_sum = 0.0f;
    constexpr float kLog2e = 1.4426950408889634f;

    // K / V tile: KEYS positions x HD floats each, in 16-byte slots
    constexpr int kSlots = KEYS * (HD / 4) / kBlock, kQpr = HD / 4;
    float4v kr[kSlots], vr[kSlots];
    typedef __attribute__((address_space(3))) char lds_char;
    lds_char *const lds = (lds_char *)pf_lds;
    constexpr uint32_t PIECE = KEYS * HD * 2; // bytes of a piece of K, and of V behind K's three
    auto load_kv = [&](uint32_t t0) {
#pragma unroll
        for (int h = 0; h < kSlots; h++) {
            // (pieces: K a row's 16 values by four lanes; V four positions of four columns)
            const uint32_t slot = tid + h * kBlock;
            const uint32_t tk = t0 + (PIECES ? tid / 4 % KEYS : slot / kQpr), dk = PIECES ? (tid / (4 * KEYS) + h * (kBlock / (4 * KEYS))) * 4 + tid % 4 : slot % kQpr;
            const uint32_t tv = t0 + (PIECES ? tid / kQpr * 4 + h : slot / kQpr), dv = PIECES ? tid % kQpr : slot % kQpr;
            kr[h] = (float4v){0.f, 0.f, 0.f, 0.f};
            vr[h] = (float4v){0.f, 0.f, 0.f, 0.f};
            if (tk < g.T) kr[h] = *reinterpret_cast<const float4v *>(g.Kc + ok + (int64_t)tk * g.k_st + dk * 4);
            if (tv < g.T) vr[h] = *reinterpret_cast<const float4v *>(g.V + ov + (int64_t)tv * g.v_st + dv * 4);
        }
    };
    auto store_kv = [&](uint32_t buf) {
        if constexpr (!PIECES) {
#pragma unroll
            for (int h = 0; h < kSlots; h++) {
                const uint32_t slot = tid + h * kBlock, t = slot / kQpr, dq = slot % kQpr;
                *reinterpret_cast<float4v *>(&Ks[buf][t][dq * 4]) = kr[h];
                *reinterpret_cast<float4v *>(&Vs[buf][t][dq * 4]) = vr[h];
            }
        } else {
            typedef __attribute__((address_space(3))) split::uint2v lds_pair;
            // K: blocks of 32 keys x 16 d in the order of the fragments' lanes (rows of the second lane group at row ^ 12)
            const uint32_t t = tid / 4 % KEYS, kg = tid % 4 / 2;
            const uint32_t k_at = (tid / (4 * KEYS) * (KEYS / 32) + t / 32) * 1024 + kg * 512 + ((t % 32) ^ (kg * 12)) * 16 + tid % 2 * 8;
            // V: blocks of 32 d x 16 keys; four rows change places by (d / 16) so that the lanes' stores cover all banks
            const uint32_t u = tid / kQpr, w = tid % kQpr, vg = u & 1;
            const uint32_t v_at = 3 * PIECE + (u / 4 * (HD / 32) + w / 8) * 1024 + vg * 512 + (u >> 1 & 1) * 8;
#pragma unroll
            for (int h = 0; h < kSlots; h++) {
                uint32_t a[3], b[3];
                split::grow(top_qk, kr[h][0], kr[h][1]);
                split::grow(top_qk, kr[h][2], kr[h][3]);
                split::split2(kr[h][0], kr[h][1], a);
                split::split2(kr[h][2], kr[h][3], b);
#pragma unroll
                for (int p = 0; p < 3; p++) *reinterpret_cast<lds_pair *>(lds + p * PIECE + k_at + h * (kBlock / (4 * KEYS)) * (KEYS / 32) * 1024) = (split::uint2v){a[p], b[p]};
            }
#pragma unroll
            for (int r = 0; r < 4; r++) {
                uint32_t a[3], b[3];
                split::grow(top_v, vr[0][r], vr[1][r]);
                split::grow(top_v, vr[2][r], vr[3][r]);
                split::split2(vr[0][r] * split::kUp, vr[1][r] * split::kUp, a);
                split::split2(vr[2][r] * split::kUp, vr[3][r] * split::kUp, b);
                const uint32_t row = (w % 8 * 4 + (r ^ (w / 4 & 3))) ^ (vg * 12);
#pragma unroll
                for (int p = 0; p < 3; p++) *reinterpret_cast<lds_pair *>(lds + p * PIECE + v_at + row * 16) = (split::uint2v){a[p], b[p]};
            }
        }
    };
    auto piece = [&](uint32_t at) { return __builtin_bit_cast(bf16x8, *reinterpret_cast<__attribute__((address_space(3))) float4v *>(lds + at)); };
    if (it_first < ntiles) { // (a part beyond the last key tile of these rows has nothing to do but to say so)
        load_kv(it_first * KEYS);
        store_kv(it_first & 1);
    }
    __syncthreads();

    for (uint32_t it = it_first; it < ntiles; it++) {
        const uint32_t cur = it & 1, t0 = it * KEYS;
        const bool more = it + 1 < ntiles;
        if (more) load_kv(t0 + KEYS);
        // ---- S^T = K Q^T for the tile: blocks of 32 keys x this wave's 32 queries
        float16v acc_s[KEYS / 32];
#pragma unroll
        for (int tb = 0; tb < KEYS / 32; tb++) {
#pragma unroll
            for (int v = 0; v < 16; v++) acc_s[tb][v] = 0.0f;
            if constexpr (PIECES) continue;
#pragma unroll
            for (int c = 0; c < (PIECES ? 0 : HD / 8); c++) {
                const float4v kf = *reinterpret_cast<const float4v *>(&Ks[cur][tb * 32 + li][c * 8 + lg * 4]);
#pragma unroll
                for (int r = 0; r < 4; r++) acc_s[tb] = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[r], qf[c][r], acc_s[tb], 0, 0, 0);
            }
        }
        if constexpr (PIECES) {
#pragma unroll
            for (int c = 0; c < HD / 16; c++)
#pragma unroll
                for (int tb = 0; tb < KEYS / 32; tb++) {
                    bf16x8 kf[3];
#pragma unroll
                    for (int p = 0; p < 3; p++) kf[p] = piece(p * PIECE + (c * (KEYS / 32) + tb) * 1024 + lg * 512 + (li ^ (lg * 12)) * 16);
#pragma unroll
                    for (int k = 0; k < 6; k++) acc_s[tb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[split::kPairA[k]], qp[c][split::kPairB[k]], acc_s[tb], 0, 0, 0);
                }
        }
        // ---- mask, running soft-max statistics of this lane's query.  Weights are 2^((x - max) log2 e) on the
        // hardware's exp2 (relative error ~1e-6 for the arguments that matter: inside the 1e-4 of element-wise math).
        // A tile that every query of the wave sees whole (the common case below the diagonal) needs no per-key test.
        const bool whole = __all((int)(live && t0 + KEYS - 1 <= iq && t0 + KEYS <= g.T));
        float tile_max = -INFINITY;
        if (whole) {
#pragma unroll
            for (int tb = 0; tb < KEYS / 32; tb++)
#pragma unroll
                for (int v = 0; v < 16; v++) tile_max = fmaxf(tile_max, acc_s[tb][v]);
        } else {
#pragma unroll
            for (int tb = 0; tb < KEYS / 32; tb++)
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    // the program's x / d + f32(i < j) * m: nothing is added to a visible key, and an invisible one
                    // (m is hugely negative: the host checks) ends with weight exp(-huge) = 0, so it is left out
                    const uint32_t t = t0 + tb * 32 + 8 * (v / 4) + 4 * lg + (v % 4);
                    const bool seen = t <= iq && t < g.T && live;
                    acc_s[tb][v] = seen ? acc_s[tb][v] : -INFINITY;
                    tile_max = fmaxf(tile_max, acc_s[tb][v]);
                }
        }
        tile_max = asf(fold_halves(asu(tile_max), LargerWords{}));
        const float new_max = fmaxf(run_max, tile_max);
        const float base = new_max == -INFINITY ? 0.0f : new_max; // a lane without a live query: keep NaN out
        const float alpha = __builtin_amdgcn_exp2f((run_max - base) * kLog2e);
        float tile_sum = 0.0f;
#pragma unroll
        for (int tb = 0; tb < KEYS / 32; tb++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const float p = __builtin_amdgcn_exp2f((acc_s[tb][v] - base) * kLog2e); // 2^-inf = 0 for a hidden key
                acc_s[tb][v] = p;
                tile_sum += p;
            }
        tile_sum = asf(fold_halves(asu(tile_sum), AddWords{}));
        run_sum = run_sum * alpha + tile_sum;
        run_max = new_max;
        if constexpr (!PIECES) {
            // ---- O^T = alpha O^T + V^T P^T: the V operand is read column-wise from the [t][d] tile (32 lanes, 32 banks)
#pragma unroll
            for (int db = 0; db < HD / 32; db++) {
#pragma unroll
                for (int v = 0; v < 16; v++) acc_o[db][v] *= alpha;
#pragma unroll
                for (int tb = 0; tb < KEYS / 32; tb++)
#pragma unroll
                    for (int q = 0; q < 4; q++) {
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            const float vf = Vs[cur][tb * 32 + q * 8 + lg * 4 + r][db * 32 + li];
                            acc_o[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(vf, acc_s[tb][q * 4 + r], acc_o[db], 0, 0, 0);
                        }
                    }
            }
        } else {
            // the tile's share of O, from zero and of negated weights every other time (split_tile.hpp)
            float16v sum[HD / 32];
            const bool odd = (it + __builtin_amdgcn_readfirstlane(wave)) % 2;
            const float up = odd ? -split::kUp : split::kUp, down = odd ? -split::kDown : split::kDown;
#pragma unroll
            for (int q = 0; q < KEYS / 16; q++) { // 16 keys: the eight weights that a lane holds of them, and V's rows in that order
                uint4w pw[3];
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    uint32_t x[3];
                    split::split2(acc_s[q / 2][q % 2 * 8 + 2 * r] * up, acc_s[q / 2][q % 2 * 8 + 2 * r + 1] * up, x);
#pragma unroll
                    for (int p = 0; p < 3; p++) pw[p][r] = x[p];
                }
#pragma unroll
                for (int db = 0; db < HD / 32; db++) {
                    bf16x8 vf[3];
                    const uint32_t row = (li ^ ((db * 2 + li / 16) & 3)) ^ (lg * 12);
#pragma unroll
                    for (int p = 0; p < 3; p++) vf[p] = piece((3 + p) * PIECE + (q * (HD / 32) + db) * 1024 + lg * 512 + row * 16);
#pragma unroll
                    for (int k = 0; k < 6; k++)
                        sum[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[split::kPairA[k]], __builtin_bit_cast(bf16x8, pw[split::kPairB[k]]),
                                                                         q || k ? sum[db] : (float16v){}, 0, 0, 0);
                }
            }
#pragma unroll
            for (int db = 0; db < HD / 32; db++)
#pragma unroll
                for (int v = 0; v < 16; v++) acc_o[db][v] = __builtin_fmaf(sum[db][v], down, acc_o[db][v] * alpha);
            __syncthreads(); // (one buffer: the tile is read)
        }
        if (more) store_kv(cur ^ 1);
        __syncthreads();
    }
    if constexpr (PIECES) {
        // (a score is a sum of products of magnitudes below 1e18: what the smallest values' pieces lose of it is nothing beside 1;
        // 64 keys' products of weights up to 1 and V, both scaled by 2^16, stay below 2^127)
        const bool bad = !(top_qk <= 1.0e18f && top_v < 0x1p88f);
        if (__syncthreads_or(bad)) return true;
    }
    if (e.ksplit > 1) { // the part's statistics and un-normalised O; lane group 0 of a wave writes the statistics
        if (live) {
            const uint64_t row = ((uint64_t)blockIdx.y * e.batch + b) * g.M + m;
            float *orow = e.part_o + row * HD;
#pragma unroll
            for (int db = 0; db < HD / 32; db++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    float4v o;
#pragma unroll
                    for (int r = 0; r < 4; r++) o[r] = acc_o[db][j * 4 + r];
                    *reinterpret_cast<float4v *>(orow + db * 32 + j * 8 + lg * 4) = o;
                }
            if (lg == 0) {
                e.part_ml[row * 2] = run_max;
                e.part_ml[row * 2 + 1] = run_sum;
            }
        }
        return false;
    }
    // ---- out[m][d] = O^T[d][m] / l[m]
    if (live) {
        uint32_t *orow = e.out + ((uint64_t)b * g.M + m) * HD;
#pragma unroll
        for (int db = 0; db < HD / 32; db++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                float4v o;
#pragma unroll
                for (int r = 0; r < 4; r++) o[r] = acc_o[db][j * 4 + r] / run_sum;
                *reinterpret_cast<float4v *>(orow + db * 32 + j * 8 + lg * 4) = o;
            }
    }
    return false;
}

template <int HD> __global__ __launch_bounds__(kBlock, HD == 64 ? 2 : 1) void prefill_attention_kernel(const AttnArgs g, const PrefillArgs e) {
    extern __shared__ float pf_lds[]; // above the static limit
    if (prefill_rows<HD, true>(g, e, pf_lds)) prefill_rows<HD, false>(g, e, pf_lds);
}

// out[row][d] = sum_p 2^((m_p - g) log2 e) O_p[row][d] / sum_p 2^((m_p - g) log2 e) l_p, g = max_p m_p: the parts of a
// prefill attention whose keys were cut over several workgroups, merged in the order of the parts.  A thread per four
// consecutive d of a row.  A part that saw no key of a row has m_p = -inf, l_p = 0 and O_p = 0: weight zero.
__global__ __launch_bounds__(kBlock) void prefill_attention_combine_kernel(const float *part_o, const float *part_ml, uint32_t *out,
                                                                           uint32_t parts, uint32_t hd, uint64_t rows) {
    const uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x, q = hd / 4;
    if (i >= rows * q) return;
    const uint64_t row = i / q;
    const uint32_t d = (uint32_t)(i % q) * 4;
    constexpr float kLog2e = 1.4426950408889634f;
    float g = -INFINITY;
    for (uint32_t p = 0; p < parts; p++) g = fmaxf(g, part_ml[((uint64_t)p * rows + row) * 2]);
    float4v num = {0.f, 0.f, 0.f, 0.f};
    float den = 0.0f;
    for (uint32_t p = 0; p < parts; p++) {
        const float *ml = part_ml + ((uint64_t)p * rows + row) * 2;
        const float w = __builtin_amdgcn_exp2f((ml[0] - g) * kLog2e);
        const float4v o = *reinterpret_cast<const float4v *>(part_o + ((uint64_t)p * rows + row) * hd + d);
        den = fmaf(w, ml[1], den);
        num[0] = fmaf(w, o[0], num[0]);
        num[1] = fmaf(w, o[1], num[1]);
        num[2] = fmaf(w, o[2], num[2]);
        num[3] = fmaf(w, o[3], num[3]);
    }
    float4v r;
#pragma unroll
    for (int k = 0; k < 4; k++) r[k] = num[k] / den;
    *reinterpret_cast<float4v *>(out + row * hd + d) = r;
}
