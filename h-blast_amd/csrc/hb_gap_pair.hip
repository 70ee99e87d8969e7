// hb_gap_pair.hip -- gfx950 kernel of the gapped extension for the usual
// subjects: up to HB_GAP_PAIR_HSPS ungapped HSPs, less than kLongSubject residues
// and bands of less than kCols columns (hb_gapped.hip takes the others).
//
// Half a wavefront owns one subject and takes its HSPs in the same order, with
// the same tests, as hb_gapped.hip; 16 of its lanes run the DP of the left side
// while the other 16 run that of the right side.  A lane holds kC neighbouring
// columns {best score, best score ending in a gap in the subject} in registers,
// so a row of four extension sides costs the scans of one row of 16 lanes (four
// DPP steps instead of six) and no LDS round trip for its cells.  Columns kCols
// to 2 kCols - 1 of the window are a second set of registers, evaluated only in
// the rows of a wavefront where a side's band reaches them.
//
// The window moves right by one lane (kC columns) when its first lane holds no
// live cell; it needs no other bookkeeping of the band:
//   * a row evaluates every column of the window.  A column right of the last
//     live one is live exactly when the sequential DP would open it (its score
//     is the row's gap score, tested against the same drop-off), and its state
//     is then the one that the sequential DP stores;
//   * a dropped cell is stored as kDead; its gap score may stay as it is, since
//     it lies below the drop-off threshold, which never falls;
//   * columns past the subject's end: letters there score kPast, and no cell of
//     a lane past the end is ever live (the window starts at a column <= 0 so
//     that the end falls between two lanes);
//   * when the last column of the window, or of the staged letters of a subject
//     longer than HB_GAP_SUBJ, is live and is not the subject's last, the band
//     may go on past it: the subject goes to the other kernel.
// Scores are kept as kBias + score + row * gap_extend: the row's term spares the
// column state's decrement (all compares of a row are between cells of that
// row), and the bias makes 0, which lane moves fill in, lower than any live cell.
//
// Bound by vector instruction issue: 120 of them per row of four sides, set-up
// included (30 a side; hb_gapped.hip spends 53 and as many scalar ones on a row
// of one side).  They fill 88% of the issue slots on the 297,173 HSPs of a
// 1,000-residue query against 2,000,000 subjects and 3/4 of them against 500,000,
// where the end of the work list weighs more.  The 73,052 HSPs of a 1,000-residue query
// against 500,000 subjects take 920 us here and 1,507 us there, the 5,191 of 350
// residues against 50,000 long-tailed subjects 186 and 340 us (950 and 195 us with
// two tests a row for the letters at hand and the last row instead of one).  One set of 6
// columns a lane took 1,000 us and left more subjects to the other kernel (373
// us of it, its longest chain of rows), 5 columns 901 and 509 us.
#include <hip/hip_runtime.h>

#include "hb_internal.h"

namespace {

constexpr int32_t kBias = 1 << 30;
constexpr int32_t kDead = 0;                // a dropped cell (they reach down to kPast - 1100)
constexpr int32_t kC = 4;                   // columns per lane and set
constexpr int32_t kCols = 16 * kC;          // columns of a set
constexpr int kWaves = 4;                   // wavefronts per workgroup
constexpr int32_t kWin = 11;                // start-point window
constexpr int32_t kLongSubject = 90000;     // subjects whose range hb_gapped.hip adjusts
constexpr uint32_t kSaved = 32;             // saved gapped HSPs per subject
constexpr int32_t kPast = -16000;           // score of a letter past the subject's end
constexpr uint32_t kPastLetter = 31;
constexpr int32_t kPad = 160;               // such letters kept on either side of a subject
static_assert(kPad >= 2 * kCols + 2 * kC + 8 && kC == 4, "letters of a window, a word a lane");
static_assert(HB_GAP_PAIR_HSPS <= 256, "order");
static_assert(kSaved <= HB_GAP_SAVED, "a subject that is left with them goes on in hb_gapped.hip");

// Lane move within 16 lanes; lanes without a source get 0, or old.
template <int CTRL>
__device__ __forceinline__ int32_t dpp(int32_t v)
{
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true);
}
template <int CTRL>
__device__ __forceinline__ int32_t dpp_old(int32_t v, int32_t old)
{
    return __builtin_amdgcn_update_dpp(old, v, CTRL, 0xf, 0xf, false);
}
constexpr int kShl1 = 0x101, kShr1 = 0x111, kBcast = 0x150;

// Two inclusive max-scans over each 16 lanes.
__device__ __forceinline__ void scan16_max2(int32_t &a, int32_t &b)
{
    a = max(a, dpp<0x111>(a));
    b = max(b, dpp<0x111>(b));
    a = max(a, dpp<0x112>(a));
    b = max(b, dpp<0x112>(b));
    a = max(a, dpp<0x114>(a));
    b = max(b, dpp<0x114>(b));
    a = max(a, dpp<0x118>(a));
    b = max(b, dpp<0x118>(b));
}

__device__ __forceinline__ uint64_t ballot(bool p) { return __builtin_amdgcn_ballot_w64(p); }
__device__ __forceinline__ bool lane_bit(uint64_t m) { return __builtin_amdgcn_inverse_ballot_w64(m); }

__device__ __forceinline__ void sync_lanes()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Per half wavefront.
struct PairLds {
    int32_t saved[6 * kSaved];   // ctx, score, q0, q1, s0, s1
    uint8_t order[HB_GAP_PAIR_HSPS];
    uint32_t subj[(2 * kPad + HB_GAP_SUBJ + 8) / 4];   // letters * 2
};
constexpr int32_t kSubjBytes = sizeof(PairLds::subj);

__global__ __launch_bounds__(kWaves * HB_WAVE) __attribute__((amdgpu_waves_per_eu(4))) void gap_pair_kernel(hb_gap_args A)
{
    __shared__ int16_t mat[32 * 32];       // scores + gap_extend
    __shared__ PairLds lds[2 * kWaves];
    const int32_t go = A.gap_open, ge = A.gap_extend, goe = go + ge;
    const int32_t X = max(A.x_dropoff, goe);
    for (int i = threadIdx.x; i < 32 * 32; i += blockDim.x)
        mat[i] = (int16_t)(((i & 31) == (int)kPastLetter ? kPast : A.mat32[i]) + ge);
    const int lane = threadIdx.x % HB_WAVE;
    const int hl = lane & 31, gl = lane & 15;
    const bool rev = (lane & 16) == 0;     // the left side runs backwards
    const int half0 = lane & 32;           // first lane of this half
    PairLds &L = lds[threadIdx.x / 32];
    uint8_t *sb = reinterpret_cast<uint8_t *>(L.subj);
    for (int i = hl; i < kSubjBytes / 4; i += 32) L.subj[i] = 0x01010101u * (2 * kPastLetter);
    __syncthreads();
    const char *mat_b = reinterpret_cast<const char *>(mat);

    // this half's bits of a mask
    auto half_bits = [&](uint64_t m) { return half0 ? (uint32_t)(m >> 32) : (uint32_t)m; };
    auto half_get = [&](int32_t v, int from) { return __shfl(v, half0 + from, HB_WAVE); };

    // The list's items are dealt to HB_QUEUES queues (item i to queue i mod
    // HB_QUEUES) and the workgroups likewise (their number is a multiple of
    // it); a half starts on an item of its own and then pops its queue (all
    // pops of one counter took 10 ns each).
    const uint32_t n_list = *A.n_list;
    const uint32_t queue = blockIdx.x % HB_QUEUES;
    const uint32_t own = gridDim.x / HB_QUEUES * (2 * kWaves);
    uint32_t next = blockIdx.x / HB_QUEUES * (2 * kWaves) + threadIdx.x / 32;
    bool first_pop = true;

    // half-uniform: the subject and its HSP under way
    bool need = true, active = true, fresh = true, ran = false, ovf = false;
    uint32_t k = 0, n = 0, r = 0, n_saved = 0, ext = 0;
    uint64_t f = 0;
    int32_t slen = 0;
    uint64_t o0 = 0;                       // the subject's place in A.res
    int32_t s_lo = 0, s_hi = 0, at0 = 0;   // its letters staged, and letter 0's place in sb
    int32_t c = 0, cut = 0, qo = 0, so = 0, ql = 0;
    // 16-lane-uniform: the side's DP
    int32_t a = 0, M = 0, N = 0, Ns = 0, top = 0, abest = 0, stop = INT32_MAX, sbase = 0;
    const uint8_t *arow = A.query;         // row a's letter at arow[a] (left: arow[-a])
    int32_t addr = 0;                      // of the letters right of the window
    // per lane
    int32_t ob[kC], ov[kC], ob2[kC], ov2[kC], sv[kC];
    int32_t colb = 0, Xl = -1;             // first column; X (-1 past the staged letters)
    uint32_t l1 = 0, l2 = 0, ln = 0;       // letters * 2 of the columns; those right of the window
    uint32_t qrow = 0, qnext = 0;          // letters * 64 of the rows to come, one per lane; letters
                                           // of the 16 rows after those
    int32_t event = 0;                     // the row after which they run out, or the last row
#pragma unroll
    for (int j = 0; j < kC; ++j) {
        ob[j] = ov[j] = ob2[j] = ov2[j] = kDead;
        sv[j] = 0;
    }
    const int32_t lane_ge = gl * kC * ge;

    // the word with the letters of the kC columns from that at `at` on (left
    // side: down from it, last letter first)
    auto letters = [&](int32_t at) {
        const int32_t q = min(max(rev ? at - 3 : at, 0), kSubjBytes - 4);
        uint32_t w;
        __builtin_memcpy(&w, sb + q, 4);
        return w;
    };
    auto ordered = [&](uint32_t w) {
        return __builtin_amdgcn_perm(0u, w, rev ? 0x00010203u : 0x03020100u);
    };
    auto row_letters = [&](int32_t a1) -> uint32_t {   // of rows a1 + gl
        const int32_t ra = min(a1 + gl, M);
        return M > 0 ? (uint32_t)(rev ? arow[-ra] : arow[ra]) : 0u;
    };

    // Stages the subject's letters [lo, hi), at most HB_GAP_SUBJ: whole aligned
    // words around them (the residues have 64 spare bytes), then the bytes
    // outside them.
    auto stage = [&](int32_t lo, int32_t hi) {
        s_lo = lo;
        s_hi = hi;
        const int32_t lead = (int32_t)((o0 + (uint32_t)lo) & 3);
        const uint32_t *src = reinterpret_cast<const uint32_t *>(A.res + (o0 + (uint32_t)lo - lead));
        const int32_t words = (hi - lo + lead + 3) >> 2;
        for (int32_t w = hl; w < words; w += 32) L.subj[kPad / 4 + w] = src[w] << 1;
        at0 = kPad + lead - lo;
        sync_lanes();
        if (hl < lead) sb[kPad + hl] = 2 * kPastLetter;
        for (int32_t i = hl; i < kPad; i += 32) sb[at0 + hi + i] = 2 * kPastLetter;
        sync_lanes();
    };

    for (;;) {
        if (need) {
            if (ran) {
                // the sides' best scores and cells
                int32_t at = INT32_MAX;
#pragma unroll
                for (int j = kC - 1; j >= 0; --j) at = sv[j] == stop ? sbase + j : at;
                for (int d = 1; d < 16; d <<= 1) at = min(at, __shfl_xor(at, d, HB_WAVE));
                const bool any = abest > 0;
                const int32_t best = any ? top - a * ge - kBias : 0;
                const int32_t bbest = any ? at : 0;
                const int32_t score = half_get(best, 0) + half_get(best, 16);
                const int32_t la = half_get(abest, 0), lb = half_get(bbest, 0);
                const int32_t ra = half_get(abest, 16), rb = half_get(bbest, 16);
                const bool right = half_get((int32_t)(M > 0 && N > 0), 16) != 0;
                if (ovf || (score >= cut && n_saved >= kSaved)) {
                    if (hl == 0) {   // hb_gapped.hip goes on with this HSP
                        A.st3[3 * (size_t)k] = r;
                        A.st3[3 * (size_t)k + 1] = ext - 1;
                        A.st3[3 * (size_t)k + 2] = n_saved;
                        A.mid[1 + atomicAdd(A.mid, 1u)] = k;
                    }
                    sync_lanes();   // (before the next pop of this half's first lane)
                    fresh = true;
                } else if (score >= cut) {
                    const int32_t q0 = ql - la, s0 = so + 1 - lb;
                    const int32_t q1 = right ? ra + qo + 1 : qo, s1 = right ? rb + so + 1 : so;
                    if (hl == 0) {
                        hb_gapped_hsp g;
                        g.oid = k;
                        g.context = c;
                        g.q_start = q0;
                        g.q_end = q1;
                        g.s_start = s0;
                        g.s_end = s1;
                        g.q_gapped_start = qo;
                        g.s_gapped_start = so;
                        g.score = score;
                        g.pad = 0;
                        A.out[f + n_saved] = g;
                        int32_t *e = L.saved + 6 * n_saved;
                        e[0] = c;
                        e[1] = score;
                        e[2] = q0;
                        e[3] = q1;
                        e[4] = s0;
                        e[5] = s1;
                    }
                    sync_lanes();
                    ++n_saved;
                }
                ++r;
                ran = false;
            }
            for (;;) {
                if (fresh) {
                    if (!first_pop) {
                        if (hl == 0)
                            next = own + atomicAdd(A.queues + HB_QUEUE_STRIDE * queue, 1u);
                        next = (uint32_t)half_get((int32_t)next, 0);
                    }
                    first_pop = false;
                    const uint64_t item = queue + (uint64_t)HB_QUEUES * next;
                    if (item >= n_list) {
                        active = false;
                        break;
                    }
                    k = A.list[item];
                    const hb_subject_stats st = A.ust[k];
                    n = st.n_hsp;
                    f = (uint64_t)st.first;
                    o0 = A.offs[k];
                    const uint64_t o1 = A.offs[k + 1];
                    if (n > HB_GAP_PAIR_HSPS || o1 - o0 >= (uint64_t)kLongSubject) {
                        if (hl == 0) A.mid[1 + atomicAdd(A.mid, 1u)] = k;
                        sync_lanes();
                        continue;
                    }
                    slen = (int32_t)(o1 - o0);
                    if (slen <= HB_GAP_SUBJ) stage(0, slen);
                    // the HSPs' order: (score desc, s_start asc, len desc, q_start asc)
                    const hb_hsp *U = A.urec + f;
                    if (n == 1) {
                        if (hl == 0) L.order[0] = 0;
                    } else {
                        for (uint32_t i0 = 0; i0 < n; i0 += 32) {
                            const uint32_t i = i0 + (uint32_t)hl;
                            const hb_hsp x = U[i < n ? i : 0];
                            uint32_t rank = 0;
                            for (uint32_t j0 = 0; j0 < n; j0 += 32) {
                                const uint32_t j = j0 + (uint32_t)hl;
                                const hb_hsp y = U[j < n ? j : 0];
                                const uint32_t nj = n - j0 < 32 ? n - j0 : 32;
                                for (uint32_t t = 0; t < nj; ++t) {
                                    const int32_t sc = half_get(y.score, (int)t);
                                    const int32_t ss = half_get(y.s_start, (int)t);
                                    const int32_t ln = half_get(y.len, (int)t);
                                    const int32_t qs = half_get(y.q_start, (int)t);
                                    const bool before =
                                        sc > x.score ||
                                        (sc == x.score &&
                                         (ss < x.s_start ||
                                          (ss == x.s_start &&
                                           (ln > x.len ||
                                            (ln == x.len &&
                                             (qs < x.q_start ||
                                              (qs == x.q_start && j0 + t < i)))))));
                                    rank += before ? 1u : 0u;
                                }
                            }
                            if (i < n) L.order[rank] = (uint8_t)i;
                        }
                    }
                    sync_lanes();
                    n_saved = ext = r = 0;
                    fresh = false;
                }
                if (r >= n) {
                    if (hl == 0) {
                        A.st3[3 * (size_t)k] = 0;
                        A.st3[3 * (size_t)k + 1] = ext;
                        A.st3[3 * (size_t)k + 2] = n_saved;
                    }
                    sync_lanes();
                    fresh = true;
                    continue;
                }
                const hb_hsp u = A.urec[f + L.order[r]];
                c = u.context;
                const int32_t base = A.ctx[c], clen = A.ctx[A.n_ctx + c];
                cut = A.ctx[2 * A.n_ctx + c];
                const uint8_t *qc = A.query + base;
                const int32_t qs = u.q_start - base, ss = u.s_start, len = u.len;
                bool in = false;
                if ((uint32_t)hl < n_saved) {
                    const int32_t *e = L.saved + 6 * hl;
                    const int32_t q0 = e[2], q1 = e[3], s0 = e[4], s1 = e[5];
                    in = e[0] == c && u.score <= e[1] && q0 <= qs && q1 >= qs && s0 <= ss &&
                         s1 >= ss && q0 <= qs + len && q1 >= qs + len && s0 <= ss + len &&
                         s1 >= ss + len;
                }
                if (half_bits(ballot(in))) {
                    ++r;
                    continue;
                }
                ++ext;
                if (slen > HB_GAP_SUBJ) {   // letters around the HSP's middle
                    const int32_t lo = max(0, min(ss + len / 2 - HB_GAP_SUBJ / 2, slen - HB_GAP_SUBJ));
                    stage(lo, lo + HB_GAP_SUBJ);
                }
                // start point: the middle of the best 11-residue window (first
                // maximum)
                if (len <= kWin) {
                    qo = qs + len / 2;
                } else {
                    int32_t best = INT32_MIN, where = 0;
                    for (int32_t e0 = kWin - 1; e0 < len; e0 += 32) {
                        const int32_t e = e0 + hl;
                        int32_t w = INT32_MIN;
                        if (e < len) {
                            w = 0;
#pragma unroll
                            for (int32_t t = 0; t < kWin; ++t) {
                                const int32_t o = e - (kWin - 1) + t;
                                const uint32_t l = slen > HB_GAP_SUBJ
                                                       ? 2u * A.res[o0 + (uint32_t)(ss + o)]
                                                       : sb[at0 + ss + o];
                                w += *reinterpret_cast<const int16_t *>(mat_b + 64 * qc[qs + o] + l);
                            }
                            w -= kWin * ge;
                        }
                        int32_t m = w;
                        for (int d = 1; d < 32; d <<= 1) m = max(m, __shfl_xor(m, d, HB_WAVE));
                        if (m > best) {
                            best = m;
                            where = e0 + (int32_t)__builtin_ctz(half_bits(ballot(e < len && w == m)));
                        }
                    }
                    qo = best > 0 ? qs + where - kWin / 2 : qs;
                }
                so = u.s_off + (qo - (u.q_off - base));
                if (so < s_lo || so >= s_hi) {   // (an HSP of more than HB_GAP_SUBJ)
                    const int32_t lo = max(0, min(so - HB_GAP_SUBJ / 2, slen - HB_GAP_SUBJ));
                    stage(lo, lo + HB_GAP_SUBJ);
                }
                // both sides' DP: row 0 holds the leading gaps within the drop-off.
                // The sequential DP has no column right of them in row 1 for the
                // last one's diagonal, so that one's score is not kept.
                ql = qo + 1;
                M = rev ? ql : clen - ql;
                N = rev ? so + 1 : slen - (so + 1);
                Ns = rev ? so + 1 - s_lo : s_hi - (so + 1);   // columns with staged letters
                arow = rev ? qc + qo + 1 : qc + qo;
                const int32_t base0 = -((kC - (Ns + 1) % kC) % kC);
                const bool some = M > 0 && N > 0;
                colb = some ? base0 + kC * gl : 0;
                Xl = some && colb <= Ns ? X : -1;
#pragma unroll
                for (int j = 0; j < kC; ++j) {
                    const int32_t b = colb + j;
                    const bool in0 = some && b >= 0 && b <= Ns && (b == 0 || goe + (b - 1) * ge <= X);
                    const int32_t v = kBias - (b ? go + b * ge : 0);
                    ob[j] = in0 && goe + b * ge <= X ? v : kDead;
                    ov[j] = in0 ? v - go : kDead;
                    ob2[j] = ov2[j] = kDead;
                }
                const int32_t org = rev ? at0 + so + 1 : at0 + so;
                const int32_t dir = rev ? -1 : 1;
                l1 = ordered(letters(org + dir * colb));
                l2 = ordered(letters(org + dir * (colb + kCols)));
                addr = org + dir * ((some ? base0 : 0) + 2 * kCols);
                ln = letters(addr);
                a = abest = 0;
                top = kBias;
                stop = INT32_MAX;
                qrow = row_letters(1) << 6;
                qnext = row_letters(17);
                event = min(16, M);
                ovf = false;
                ran = true;
                break;
            }
        }
        const uint64_t act = ballot(active);
        if (act == 0) break;
        const bool cut_off = ballot(Ns < N) != 0;   // some side's letters end before its subject

        // One row of a set of columns: the cells' new states, the masks of its
        // live cells and of those in the lanes' last column, its largest score.
        // left: the previous row's score left of its first column per lane; ca, cb:
        // the earlier columns' largest U and score.  All T and U stay below those
        // of the last lane (total_*).
        struct Row {
            uint64_t any, last;
            int32_t S[kC], total_u, total_t;
        };
        auto eval = [&](const char *mrow, uint32_t l, int32_t left, int32_t col_ge, int32_t lim,
                        int32_t ca, int32_t cb, int32_t *o, int32_t *v) {
            Row w;
            int32_t T[kC], U[kC];
#pragma unroll
            for (int j = 0; j < kC; ++j)
                T[j] = *reinterpret_cast<const int16_t *>(mrow + ((l >> (8 * j)) & 255u));
#pragma unroll
            for (int j = 0; j < kC; ++j) T[j] = max((j ? o[j - 1] : left) + T[j], v[j]);
            // U(j) = T(j) + column * ge, from which the gap score of the columns
            // to the right follows
            int32_t ia = INT32_MIN, ib = INT32_MIN;
#pragma unroll
            for (int j = 0; j < kC; ++j) {
                U[j] = T[j] + col_ge + j * ge;
                ia = max(ia, U[j]);
                ib = max(ib, T[j]);
            }
            scan16_max2(ia, ib);
            w.total_u = ia;
            w.total_t = dpp<kBcast + 15>(ib);
            int32_t pa = max(dpp<kShr1>(ia), ca);
            int32_t pb = max(dpp<kShr1>(ib), cb);
            w.any = 0;
#pragma unroll
            for (int j = 0; j < kC; ++j) {
                const int32_t R = pa - col_ge - (goe - ge + j * ge);
                w.S[j] = max(T[j], R);
                w.last = ballot(pb - w.S[j] <= lim);
                w.any |= w.last;
                o[j] = lane_bit(w.last) ? w.S[j] : kDead;
                v[j] = max(w.S[j] - go, v[j]);
                pa = max(pa, U[j]);
                pb = max(pb, T[j]);
            }
            return w;
        };
        constexpr uint64_t kLane15 = 0x8000800080008000ull, kLane0 = 0x0001000100010001ull;

        // rows of all sides under way, until both sides of a half are done
        uint64_t live;
        bool wide = true;   // some side's second set may hold live cells
        do {
            ++a;
            top += ge;
            const int32_t row = dpp<kBcast>((int32_t)qrow);
            qrow = (uint32_t)dpp<kShl1>((int32_t)qrow);
            const char *mrow = mat_b + row;
            const int32_t last_ob = ob[kC - 1];
            const Row w = eval(mrow, l1, dpp<kShr1>(last_ob), lane_ge, Xl, 0, top, ob, ov);
            live = w.any;
            uint64_t live0 = w.any;     // of the first set
            uint64_t over = 0;
            int32_t rmax = w.total_t;   // the row's best score
            if (wide || (w.last & kLane15)) {
                const int32_t left = dpp_old<kShr1>(ob2[kC - 1], dpp<kBcast + 15>(last_ob));
                const Row w2 = eval(mrow, l2, left, lane_ge + kCols * ge,
                                    colb + kCols <= Ns ? X : -1, dpp<kBcast + 15>(w.total_u),
                                    max(rmax, top), ob2, ov2);
                wide = (w2.any | (w.last & kLane15)) != 0;
                live |= w2.any;
                if (w2.last & kLane15) over = ballot(colb + kCols + kC <= N) & w2.last & kLane15;
                if (cut_off) over |= ballot(Ns < N && colb + kCols + kC - 1 == Ns) & w2.last;
                // the row's best cell is in the second set when that exceeds the first's
                if (w2.total_t > max(rmax, top)) {
                    top = stop = w2.total_t;
                    abest = a;
                    sbase = colb + kCols;
#pragma unroll
                    for (int j = 0; j < kC; ++j) sv[j] = w2.S[j];
                }
            }
            if (cut_off) over |= ballot(Ns < N && colb + kC - 1 == Ns) & w.last;
            const uint64_t up = ballot(rmax > top);
            if (up) {
                if (lane_bit(up)) {
                    top = stop = rmax;
                    abest = a;
                    sbase = colb;
#pragma unroll
                    for (int j = 0; j < kC; ++j) sv[j] = w.S[j];
                }
            }
            // the rows, or the letters at hand, are used up
            if (ballot(a == event)) {
                const uint64_t end = ballot(a == event && a == M);
                live &= ~end;
                live0 &= ~end;
#pragma unroll
                for (int j = 0; j < kC; ++j) {
                    ob[j] = lane_bit(end) ? kDead : ob[j];
                    ov[j] = lane_bit(end) ? kDead : ov[j];
                    ob2[j] = lane_bit(end) ? kDead : ob2[j];
                    ov2[j] = lane_bit(end) ? kDead : ov2[j];
                }
                if (a == event) {
                    event = min(a + 16, M);
                    qrow = qnext << 6;
                    qnext = row_letters(a + 17);
                }
            }
            // the band may leave the window, or the staged letters
            over &= live;
            if (over) {
                uint64_t gone = 0;
                if (over & 0xffffffffull) gone |= 0xffffffffull;
                if (over >> 32) gone |= 0xffffffff00000000ull;
                ovf = ovf || lane_bit(gone);
                live &= ~gone;
                live0 &= ~gone;
#pragma unroll
                for (int j = 0; j < kC; ++j) {
                    ob[j] = lane_bit(gone) ? kDead : ob[j];
                    ov[j] = lane_bit(gone) ? kDead : ov[j];
                    ob2[j] = lane_bit(gone) ? kDead : ob2[j];
                    ov2[j] = lane_bit(gone) ? kDead : ov2[j];
                }
            }
            // no live cell in a side's first lane: its window moves by one lane
            const uint64_t z = ~live0 & kLane0;
            if (z) {
                if (lane_bit((z << 16) - z)) {
                    if (wide) {
#pragma unroll
                        for (int j = 0; j < kC; ++j) {
                            ob[j] = dpp_old<kShl1>(ob[j], dpp<kBcast>(ob2[j]));
                            ov[j] = dpp_old<kShl1>(ov[j], dpp<kBcast>(ov2[j]));
                            ob2[j] = dpp<kShl1>(ob2[j]);
                            ov2[j] = dpp<kShl1>(ov2[j]);
                        }
                    } else {
#pragma unroll
                        for (int j = 0; j < kC; ++j) {
                            ob[j] = dpp<kShl1>(ob[j]);
                            ov[j] = dpp<kShl1>(ov[j]);
                        }
                    }
                    l1 = (uint32_t)dpp_old<kShl1>((int32_t)l1, dpp<kBcast>((int32_t)l2));
                    l2 = (uint32_t)dpp_old<kShl1>((int32_t)l2, (int32_t)ordered(ln));
                    colb += kC;
                    Xl = colb <= Ns ? Xl : -1;
                    addr += rev ? -kC : kC;
                    ln = letters(addr);
                }
            }
            const uint64_t run = live | ~act;
            if ((uint32_t)run == 0 || (uint32_t)(run >> 32) == 0) break;
        } while (true);
        need = active && half_bits(live) == 0;
    }
}

}  // namespace

hipError_t hb_launch_gap_pair(const hb_gap_args &a, int n_blocks, hipStream_t st)
{
    if (n_blocks < HB_QUEUES || n_blocks % HB_QUEUES) return hipErrorInvalidValue;
    hipLaunchKernelGGL(gap_pair_kernel, dim3(n_blocks), dim3(kWaves * HB_WAVE), 0, st, a);
    return hipGetLastError();
}

bool hb_gap_pair_ok(int32_t gap_open, int32_t gap_extend, int32_t x_dropoff)
{
    if (gap_extend < 1 || gap_extend > 100 || gap_open > 1000) return false;
    const int32_t goe = gap_open + gap_extend, X = x_dropoff > goe ? x_dropoff : goe;
    // The drop-off stays below kPast.  Bands grow to 1.9 times row 0's on average
    // and 3.4 times at most (8,038 extensions with the default parameters), so
    // that a row 0 of a quarter of the window leaves nearly none to the other
    // kernel, whose longest chain of rows then comes on top (270 us where 20 of
    // 55,000 subjects were left to it).
    return X <= -kPast / 2 && (X - goe) / gap_extend + 2 <= 2 * kCols / 4;
}
