// bitpar.hip -- gfx950 bit-parallel aligner for pairs of many edits.
//
// The wavefront search of kernels.hip costs a cell per (level, diagonal), about
// D*D/2 for a pair of distance D.  Here the same alignment comes out of the
// edit-distance table itself, 32 rows of a column per 32-bit word as vertical
// delta bits (Myers' bit vectors, in Hyyro's form), over a band of diagonals:
// about 0.5 instruction per table cell and lane, so a pair of n bases costs
// n * D * 0.5 against the wavefront's D * D * 15, and from some 3 to 4 percent of
// edits on this is the cheaper of the two.
//
// Distance and CIGAR are the wavefront's, bit for bit.  The wavefront's
// traceback takes, at a cell of diagonal k and level d, the candidate that lands
// furthest on the diagonal (DEL, then SUB, then INS on ties; src/kernels.cu:141-152).
// Walking the diagonal back from the furthest cell of value d, that is the first
// cell whose upper neighbour has value d-1 (DEL), else whose diagonal neighbour
// has (SUB), else whose left neighbour has (INS): a candidate with a larger
// offset would have been met earlier.  So the path is read off the table's
// deltas: DEL where the vertical delta is +1, else SUB where the diagonal delta
// is +1, else INS where the horizontal delta is +1, else a match.
//
// A band that holds every diagonal a path of at most L edits can touch
// (-floor((L-tk)/2) .. floor((L+tk)/2), tk the target diagonal) gives exact values
// on all such paths, and values no lower than the table's elsewhere: outside
// values enter as +1 deltas, which are upper bounds.  A path found with at most L
// edits is therefore the path; a pair that takes more is deferred.
#include "device.h"
#include "ewfa_internal.h"

namespace ewfa {

namespace {

// Lanes of each group of GL that start one.
template <int GL>
__host__ __device__ constexpr uint64_t group_starts() {
    uint64_t m = 0;
    for (int i = 0; i < 64; i += GL) m |= 1ull << i;
    return m;
}

// The 32 bases of a packed word as two bit planes, base i in bit i of both.
__device__ __forceinline__ void planes_of(uint64_t w, uint32_t& a, uint32_t& b) {
    // bit-reversed, base i sits in bits 2i, 2i+1; the even bits of a 64-bit
    // word move together in five steps of 32-bit halves
    const uint64_t r = __builtin_bitreverse64(w);
    const auto even = [](uint32_t x) -> uint32_t {
        x &= 0x55555555u;
        x = (x | (x >> 1)) & 0x33333333u;
        x = (x | (x >> 2)) & 0x0F0F0F0Fu;
        x = (x | (x >> 4)) & 0x00FF00FFu;
        return (x | (x >> 8)) & 0xFFFFu;
    };
    const uint32_t lo = (uint32_t)r, hi = (uint32_t)(r >> 32);
    a = even(lo) | (even(hi) << 16);
    b = even(lo >> 1) | (even(hi >> 1) << 16);
}

// A lane's value from the lane before it in its group of GL, 0 in a group's
// first lane.
template <int GL>
__device__ __forceinline__ uint32_t from_above(uint32_t x, int lane) {
    // row_shr:1 within rows of 16 lanes, else wave_shr:1
    const uint32_t y = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, GL <= 16 ? 0x111 : 0x138, 0xF, 0xF, true);
    if constexpr (GL == 64 || GL == 16) return y;
    return y & ((lane & (GL - 1)) ? ~0u : 0u);
}

// A lane's value from the lane after it in its group; a group's last lane
// gets `bottom`.
template <int GL>
__device__ __forceinline__ uint32_t from_below(uint32_t x, uint32_t bottom, int lane) {
    // row_shl:1 or wave_shl:1
    const uint32_t y =
        (uint32_t)__builtin_amdgcn_update_dpp((int)bottom, (int)x, GL <= 16 ? 0x101 : 0x130, 0xF, 0xF, false);
    if constexpr (GL == 64 || GL == 16) return y;
    return (lane & (GL - 1)) == GL - 1 ? bottom : y;
}

// A lane's value from lane x (uniform) of its group.
template <int GL>
__device__ __forceinline__ uint32_t from_group(uint32_t v, int x, int lane) {
    if constexpr (GL == 64) return (uint32_t)__builtin_amdgcn_readlane((int)v, x);
    return (uint32_t)__builtin_amdgcn_ds_bpermute(((lane & ~(GL - 1)) + x) << 2, (int)v);
}

// Inclusive sum, minimum and maximum over a group.
template <int GL>
__device__ __forceinline__ int group_incl_sum(int v, int lane) {
#pragma unroll
    for (int d = 1; d < GL; d <<= 1) {
        const int t = __builtin_amdgcn_ds_bpermute((lane - d) << 2, v);
        if ((lane & (GL - 1)) >= d) v += t;
    }
    return v;
}
template <int GL>
__device__ __forceinline__ int group_max(int v, int lane) {
#pragma unroll
    for (int d = 1; d < GL; d <<= 1) v = max(v, (int)__builtin_amdgcn_ds_bpermute((lane ^ d) << 2, v));
    return v;
}

struct BpPair {
    const uint64_t* gp;  // packed words
    const uint64_t* gt;
    int plen, tlen, nwp, nwt, tk;
    int L;               // the most edits looked for
    int S;               // band: words j + S .. at column block j
};

// The band's widths over the column blocks: segment k starts at block
// from[k], with w[k] words a lane, its records from row at[k] on (a row: 64
// lanes of Pv, Mv, then 64 lanes of the horizontal deltas below the word).
// Uniform over the wave; S[k] is each pair's own.
struct BpSegs {
    int from[4], w[4], at[4], S[4];
};

__device__ __forceinline__ BpPair bp_load(const BpArgs& a, uint32_t pidx, const ewfa_pair_t& pr, int N) {
    BpPair p;
    p.gp = a.words + pr.pattern_off;
    p.gt = a.words + pr.text_off;
    p.plen = (int)pr.plen;
    p.tlen = (int)pr.tlen;
    p.nwp = (p.plen + 31) >> 5;
    p.nwt = (p.tlen + 31) >> 5;
    p.tk = p.tlen - p.plen;
    p.L = min(bp_band(N, p.tk, p.S), (int)min(a.bound[pidx], 0x7FFFFFFFu));
    return p;
}

// x + y over W words, first word lowest: the sums, the lanes whose top word
// overflows (G) and the lanes whose words are all ones (P).  A carry read by the
// vector unit two instructions or less after it wrote it would need the wait
// states here.
template <int W>
__device__ __forceinline__ void add_words(const uint32_t (&x)[W], const uint32_t (&y)[W], uint32_t (&s)[W],
                                          uint64_t& G, uint64_t& P) {
    if constexpr (W == 1) {
        asm("v_add_co_u32_e64 %0, %1, %3, %4\n\t"
            "v_cmp_eq_u32_e64 %2, -1, %0"
            : "=&v"(s[0]), "=&s"(G), "=s"(P)
            : "v"(x[0]), "v"(y[0]));
    } else {
        uint64_t c;
        asm("v_add_co_u32_e64 %0, %1, %2, %3" : "=v"(s[0]), "=s"(c) : "v"(x[0]), "v"(y[0]));
        uint32_t ones = s[0];
#pragma unroll
        for (int w = 1; w < W; ++w) {
            asm("s_nop 1\n\tv_addc_co_u32_e64 %0, %1, %2, %3, %4"
                : "=v"(s[w]), "=s"(G)
                : "v"(x[w]), "v"(y[w]), "s"(c));
            c = G;
            ones &= s[w];
        }
        asm("v_cmp_eq_u32_e64 %0, -1, %1" : "=s"(P) : "v"(ones));
    }
}

// s + carry (a lane mask) over W words.
template <int W>
__device__ __forceinline__ void add_carry(uint32_t (&s)[W], uint64_t cin) {
    uint64_t c;
    asm("v_addc_co_u32_e64 %0, %1, 0, %0, %2" : "+v"(s[0]), "=&s"(c) : "s"(cin));
#pragma unroll
    for (int w = 1; w < W; ++w) {
        const uint64_t b = c;
        asm("s_nop 1\n\tv_addc_co_u32_e64 %0, %1, 0, %0, %2" : "+v"(s[w]), "=&s"(c) : "s"(b));
    }
}

// One column of the band: W words per lane, GL lanes per pair, every lane of
// the wave taking part.  c0, c1: the text base's bits as masks.  nhp, hm gather
// the horizontal deltas below each word (nhp: those that are not +1).  19
// vector instructions at W = 1, 14 to 16 per word more.
template <int GL, int W>
__device__ __forceinline__ void bp_column(uint32_t (&Pv)[W], uint32_t (&Mv)[W], const uint32_t (&P0)[W],
                                          const uint32_t (&P1)[W], uint32_t c0, uint32_t c1,
                                          uint32_t (&nhp)[W], uint32_t (&hm)[W], int lane) {
    uint32_t Eq[W], x[W], s[W];
#pragma unroll
    for (int w = 0; w < W; ++w) {
        Eq[w] = ~(P0[w] ^ c0) & ~(P1[w] ^ c1);
        x[w] = Eq[w] & Pv[w];
    }
    // carries between lanes: a lane that overflows (G) hands one to the next,
    // a lane of all ones (P) passes one on; one 64-bit scalar addition finds
    // every lane's carry in
    uint64_t G, P;
    add_words<W>(x, Pv, s, G, P);
    uint64_t g1 = G << 1;
    if constexpr (GL < 64) {
        g1 &= ~group_starts<GL>();
        P &= ~(group_starts<GL>() << (GL - 1));
    }
    add_carry<W>(s, (P + g1) ^ P);
    uint32_t nPh[W], Mh[W];  // horizontal deltas: not +1, -1
#pragma unroll
    for (int w = 0; w < W; ++w) {
        const uint32_t Xh = (s[w] ^ Pv[w]) | Eq[w];
        nPh[w] = ~Mv[w] & (Xh | Pv[w]);
        Mh[w] = Pv[w] & Xh;
    }
#pragma unroll
    for (int w = 0; w < W; ++w) {
        nhp[w] = __builtin_amdgcn_alignbit(nhp[w], nPh[w], 31);
        hm[w] = __builtin_amdgcn_alignbit(hm[w], Mh[w], 31);
    }
    const uint32_t pd = from_above<GL>(nPh[W - 1], lane);  // +1 above the band's first row
    const uint32_t md = from_above<GL>(Mh[W - 1], lane);
#pragma unroll
    for (int w = W - 1; w >= 0; --w) {
        const uint32_t ps = __builtin_amdgcn_alignbit(nPh[w], w ? nPh[w ? w - 1 : 0] : pd, 31);
        const uint32_t ms = __builtin_amdgcn_alignbit(Mh[w], w ? Mh[w ? w - 1 : 0] : md, 31);
        const uint32_t Xv = Eq[w] | Mv[w];
        Pv[w] = ms | (ps & ~Xv);
        Mv[w] = Xv & ~ps;
    }
}

// One segment of the table's deltas of 64/GL pairs (p: the lane's own), from
// column block j on in blocks of 32 columns: until nblk, or until no pair of
// the wave needs more than `fewer` words a lane (looked at every BP_LOOK blocks;
// then the band moves to the words still needed and `w` says how many words a
// lane they take).  Records every block's deltas (BpSegs) at rec.
//
// What a pair still needs: a cell (v, h) of value D on diagonal k is on a path of
// at most L edits only if D + |k - tk| <= L, and such a path stays on diagonals
// min(k, tk) - s/2 .. max(k, tk) + s/2 from there on, s = L - D - |k - tk|.  Values
// are looked at where words meet; a cell up to 16 rows away has s at most 32
// larger, which the range takes in.  A band that started U wide narrows to
// nothing about linearly, so half of the table is never computed.
constexpr int BP_LOOK = 8;

// A narrowed band's words pass from one segment to the next in LDS, 4 planes of
// n_prev words a group, this band's from `first` on (n_prev 0: the first segment).
template <int GL, int W>
__device__ __forceinline__ int bp_segment(BpPair& p, int j, int nblk, int& n_prev, int& first, int& sc, uint2*& rec,
                                          int& w_next, uint32_t* lds, int lane) {
    constexpr int N = GL * W;
    const int gl = lane & (GL - 1);
    uint32_t vp[W], vm[W], q0[W], q1[W];
    if (n_prev) {
        const uint32_t* G = lds + (lane / GL) * (4 * n_prev) + first + gl * W;
        group_sync<1>();
#pragma unroll
        for (int w = 0; w < W; ++w) {
            vp[w] = G[w];
            vm[w] = G[n_prev + w];
            q0[w] = G[2 * n_prev + w];
            q1[w] = G[3 * n_prev + w];
        }
        group_sync<1>();
    } else {
#pragma unroll
        for (int w = 0; w < W; ++w) {
            // rows above the first (negative words) count down to it, so that
            // row 0 holds h in every column whatever their bases
            const int A = p.S + gl * W + w;
            vp[w] = A < 0 ? 0u : ~0u;
            vm[w] = A < 0 ? ~0u : 0u;
            planes_of(p.gp[min(max(A, 0), p.nwp)], q0[w], q1[w]);
        }
    }
    int x = GL;  // feeder place
    uint32_t f0 = 0, f1 = 0, e0 = 0, e1 = 0;
    const int j0 = j;
    w_next = W;
    for (; j < nblk; ++j) {
        if (x == GL) {
            // the next GL blocks' text planes and the pattern planes that enter
            // the band with them, one per lane
            planes_of(p.gt[min(j + gl, p.nwt)], f0, f1);
            planes_of(p.gp[min(max(j + gl + p.S + N - 1, 0), p.nwp)], e0, e1);
            x = 0;
        }
        if (j > j0) {  // the band moves down a word
            sc += 32 + __popc(vp[0]) - __popc(vm[0]);  // (a group's first lane: the value above its band)
            const uint32_t b0 = from_below<GL>(vp[0], ~0u, lane);
            const uint32_t b1 = from_below<GL>(vm[0], 0u, lane);
            const uint32_t b2 = from_below<GL>(q0[0], from_group<GL>(e0, x, lane), lane);
            const uint32_t b3 = from_below<GL>(q1[0], from_group<GL>(e1, x, lane), lane);
#pragma unroll
            for (int w = 0; w + 1 < W; ++w) {
                vp[w] = vp[w + 1];
                vm[w] = vm[w + 1];
                q0[w] = q0[w + 1];
                q1[w] = q1[w + 1];
            }
            vp[W - 1] = b0;
            vm[W - 1] = b1;
            q0[W - 1] = b2;
            q1[W - 1] = b3;
            if (W > 1 && ((j - j0) % BP_LOOK) == 0) {
                // values where words meet, and the diagonals still in reach
                int tot = 0;
#pragma unroll
                for (int w = 0; w < W; ++w) tot += __popc(vp[w]) - __popc(vm[w]);
                int D = (int)from_group<GL>((uint32_t)sc, 0, lane) + group_incl_sum<GL>(tot, lane) - tot;
                int lo = 1 << 28, hi = -(1 << 28);  // first and last diagonals
                const auto look = [&](int k, int d) {
                    const int sl = p.L - d - abs(k - p.tk);
                    if (sl + 32 >= 0) {
                        const int ext = ((sl + 1) >> 1) + 32;
                        lo = min(lo, min(k, p.tk) - ext);
                        hi = max(hi, max(k, p.tk) + ext);
                    }
                };
                if (gl == 0) look(-32 * p.S, D);
#pragma unroll
                for (int w = 0; w < W; ++w) {
                    D += __popc(vp[w]) - __popc(vm[w]);
                    look(-32 * (p.S + gl * W + w + 1), D);
                }
                hi = group_max<GL>(hi, lane);
                lo = -group_max<GL>(-lo, lane);
                // word i holds diagonals -32(S+i)-31 .. -32(S+i)+31
                const int ia = min(max(((-hi) >> 5) - p.S, 0), N);
                const int ib = max(min(((31 - lo) >> 5) + 1 - p.S, N), 0);
                const int need = max(ib - ia, 1);
                const int wn = (need + GL - 1) / GL;
                // the wave's pairs go on together: the most any needs
                int most = 1;
#pragma unroll
                for (int v = W; v >= 2; --v)
                    if (most == 1 && __builtin_amdgcn_ballot_w64(wn >= v && j < p.nwt)) most = v;
                if (most < W) {
                    w_next = most;
                    first = min(ia, N - GL * most);
                    n_prev = N;
                    uint32_t* G = lds + (lane / GL) * (4 * N);
                    group_sync<1>();
#pragma unroll
                    for (int w = 0; w < W; ++w) {
                        const int at = gl * W + w;
                        G[at] = vp[w];
                        G[N + at] = vm[w];
                        G[2 * N + at] = q0[w];
                        G[3 * N + at] = q1[w];
                    }
                    group_sync<1>();
                    int drop = 0;  // deltas of the words dropped at the top
                    for (int i = gl; i < first; i += GL) drop += __popc(G[i]) - __popc(G[N + i]);
                    drop = group_incl_sum<GL>(drop, lane);
                    sc += (int)from_group<GL>((uint32_t)drop, GL - 1, lane);
                    p.S += first;
                    return j;
                }
            }
        }
        uint32_t T0 = from_group<GL>(f0, x, lane), T1 = from_group<GL>(f1, x, lane);
        ++x;
#pragma unroll
        for (int w = 0; w < W; ++w) rec[w * 128 + lane] = make_uint2(vp[w], vm[w]);
        uint32_t nhp[W], hm[W];
#pragma unroll
        for (int w = 0; w < W; ++w) nhp[w] = hm[w] = 0;
        for (int i8 = 0; i8 < 32; i8 += 8) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint32_t c0 = (uint32_t)((int)(T0 << (31 - i)) >> 31);
                const uint32_t c1 = (uint32_t)((int)(T1 << (31 - i)) >> 31);
                bp_column<GL, W>(vp, vm, q0, q1, c0, c1, nhp, hm, lane);
            }
            T0 >>= 8;
            T1 >>= 8;
        }
#pragma unroll
        for (int w = 0; w < W; ++w) rec[w * 128 + 64 + lane] = make_uint2(~nhp[w], hm[w]);
        rec += W * 128;
    }
    return j;
}

// The whole table: segments of decreasing width.
template <int GL>
__device__ __forceinline__ void bp_forward(BpPair p, int W, int nblk, uint2* rec, BpSegs& sg, uint32_t* lds,
                                           int lane) {
    int sc = -32 * p.S, j = 0, w = W, n_prev = 0, first = 0;
    const uint2* const rec0 = rec;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        sg.from[k] = 0x7FFFFFFF;
        sg.w[k] = 1;
        sg.at[k] = 0;
        sg.S[k] = 0;
        if (j >= nblk) continue;
        sg.from[k] = j;
        sg.w[k] = w;
        sg.at[k] = (int)((rec - rec0) >> 7);
        sg.S[k] = p.S;
        int wn = w;
        if (w == 4) j = bp_segment<GL, 4>(p, j, nblk, n_prev, first, sc, rec, wn, lds, lane);
        else if (w == 3) j = bp_segment<GL, 3>(p, j, nblk, n_prev, first, sc, rec, wn, lds, lane);
        else if (w == 2) j = bp_segment<GL, 2>(p, j, nblk, n_prev, first, sc, rec, wn, lds, lane);
        else j = bp_segment<GL, 1>(p, j, nblk, n_prev, first, sc, rec, wn, lds, lane);
        w = wn;
    }
}

// ---- traceback ---------------------------------------------------------------
// The paths are walked back over tiles of 32 rows x 32 columns whose op codes
// are computed again from the recorded deltas, a lane a tile: TW row words
// around the path's diagonal over TB column blocks.  The codes (two bits a cell,
// equal to OP_*, 0 for a match) go to LDS, where lanes look along the diagonal at
// once, each at a cell so many steps back, so a match run and the op that ends
// it are one step.
// Bands of 16 lanes and less (bp_walk): the wave's groups walk side by side, a
// group over its own GL tiles, and take new tiles together.
// Wider bands (bp_walk_wave): one pair after the other, the whole wave looking 64
// cells back and the walk itself in scalar registers.
template <int GL>
struct TraceShape {
    static constexpr int TW = GL >= 32 ? 4 : 2, TB = GL >= 32 ? 8 : GL / TW, RL = 16;
    static constexpr int TILES = GL >= 32 ? TW * TB : 64;  // of the wave
};
// uint2 per tile; column c of tile t at c ^ tile_swizzle(t), which keeps pairs of
// columns together and spreads the tiles over the banks
constexpr int TILE_WORDS = 32;
__device__ __forceinline__ int tile_swizzle(int t) { return (t & 15) << 1; }

// Codes of one tile: pv, mv the word's deltas before the block, h the
// horizontal deltas above it, p0, p1 and T0, T1 the pattern's and text's planes.
__device__ __forceinline__ void trace_tile(uint32_t pv, uint32_t mv, uint2 h, uint32_t p0, uint32_t p1, uint32_t T0,
                                           uint32_t T1, uint2* out, int swz) {
    const auto column = [&](int i) -> uint2 {
        const uint32_t c0 = (uint32_t)((int)(T0 << (31 - i)) >> 31);
        const uint32_t c1 = (uint32_t)((int)(T1 << (31 - i)) >> 31);
        const uint32_t E = ~(p0 ^ c0) & ~(p1 ^ c1);
        const uint32_t Xv = E | mv;
        const uint32_t Eq = E | (h.y >> 31);
        const uint32_t Xh = (((Eq & pv) + pv) ^ pv) | Eq;
        const uint32_t Ph = mv | ~(Xh | pv), Mh = pv & Xh;
        const uint32_t D0 = Xh | mv;  // diagonal delta 0
        const uint32_t ps = __builtin_amdgcn_alignbit(Ph, h.x, 31), ms = __builtin_amdgcn_alignbit(Mh, h.y, 31);
        h.x <<= 1;
        h.y <<= 1;
        pv = ms | ~(Xv | ps);
        mv = ps & Xv;
        // DEL 3: vertical +1; else SUB 2: diagonal +1; else INS 1: horizontal +1
        const uint32_t hi = pv | ~D0;
        return make_uint2(hi, pv | (Ph & ~hi));
    };
#pragma unroll 4
    for (int i = 0; i < 32; i += 2) {
        const uint2 a = column(i), b = column(i + 1);
        *reinterpret_cast<uint4*>(out + (i ^ swz)) = make_uint4(a.x, a.y, b.x, b.y);
    }
}

// A group's bits of a wave mask.
template <int GL>
__device__ __forceinline__ uint64_t group_bits(uint64_t m, int lane) {
    if constexpr (GL == 64) return m;
    const uint32_t half = lane < 32 ? (uint32_t)m : (uint32_t)(m >> 32);
    if constexpr (GL == 32) return half;
    return (half >> (lane & 31 & ~(GL - 1))) & ((1u << GL) - 1u);
}

// The tile (block J, word idx of the band there) into `out`; S, w, at: the band of
// J's segment; lane0: the group's first lane.
__device__ __forceinline__ void bp_tile(const BpPair& p, const uint2* rec, int J, int idx, int S, int w, int at,
                                        int lane0, uint2* out, int swz) {
    const int l = (int)((unsigned)idx / (unsigned)w), x = idx - l * w;
    const uint2 d = rec[(size_t)(at + x) * 128 + lane0 + l];
    uint2 h = make_uint2(~0u, 0u);  // +1 above the band
    if (idx > 0) h = rec[(size_t)(at + (x ? x - 1 : w - 1)) * 128 + 64 + lane0 + (x ? l : l - 1)];
    uint32_t p0, p1, T0, T1;
    planes_of(p.gp[min(max(J + S + idx, 0), p.nwp)], p0, p1);
    planes_of(p.gt[min(J, p.nwt)], T0, T1);
    trace_tile(d.x, d.y, h, p0, p1, T0, T1, out, swz);
}

// The segment of block J: its band's first word S, words a lane w and J's first
// record row `at`.
__device__ __forceinline__ void bp_segment_of(const BpSegs& sg, int J, int& S, int& w, int& at) {
    w = sg.w[0];
    S = sg.S[0];
    at = sg.at[0] + (J - sg.from[0]) * w;
#pragma unroll
    for (int k = 1; k < 4; ++k)
        if (J >= sg.from[k]) {
            w = sg.w[k];
            S = sg.S[k];
            at = sg.at[k] + (J - sg.from[k]) * w;
        }
}

// The path of one pair, p and sg uniform, as bp_walk gives it.
template <int GL>
__device__ __forceinline__ int bp_walk_wave(const BpPair& p, const BpSegs& sg, int lane0, const uint2* rec,
                                            uint32_t* tok, uint2* tiles, int& run, int lane) {
    typedef TraceShape<GL> T;
    int rho = p.plen - 1, gam = p.tlen - 1;  // the cell's row and column, from 0
    int cnt = 0, tokv = 0;
    run = 0;
    const auto push = [&](int op) {
        tokv = writelane_i32(tokv, (run << 2) | op, cnt & 63);
        run = 0;
        ++cnt;
        if ((cnt & 63) == 0) tok[cnt - 64 + lane] = (uint32_t)tokv;
    };
    if (p.L < 0) return -1;
    int j0 = 0, base = 0;
    uint64_t tm = 0;  // tiles that lie in the band
    bool have = false;
    while (rho >= 0 && gam >= 0) {
        const bool fresh = !have;
        if (!have) {
            j0 = gam >> 5;
            base = (rho - gam - 32) >> 5;  // the path's diagonal in the middle words
            const int t = lane & (T::TILES - 1);
            const int J = j0 - t / T::TW;
            int S, w, at;
            bp_segment_of(sg, J, S, w, at);
            const int idx = base + t % T::TW - S;
            const bool in = J >= 0 && idx >= 0 && idx < GL * w;
            tm = __builtin_amdgcn_ballot_w64(in);
            group_sync<1>();
            if (in && lane < T::TILES) bp_tile(p, rec, J, idx, S, w, at, lane0, tiles + t * TILE_WORDS, tile_swizzle(t));
            group_sync<1>();
            have = true;
        }
        const int r = rho - lane, g = gam - lane;
        const int Jc = g >> 5, q = j0 - Jc, u = (r >> 5) - Jc - base, t = q * T::TW + u;
        const bool in = r >= 0 && g >= 0 && q < T::TB && (unsigned)u < (unsigned)T::TW && ((tm >> (t & 63)) & 1u);
        const uint2 cc = tiles[in ? t * TILE_WORDS + ((g & 31) ^ tile_swizzle(t)) : 0];
        const uint64_t hib = __builtin_amdgcn_ballot_w64(in && ((cc.x >> (r & 31)) & 1u));
        const uint64_t lob = __builtin_amdgcn_ballot_w64(in && ((cc.y >> (r & 31)) & 1u));
        const uint64_t out = __builtin_amdgcn_ballot_w64(!in);
        const uint64_t stop = hib | lob | out;
        if (fresh && (out & 1ull)) return -1;  // outside the band: more than L edits
        int pos = 0;
        for (;;) {
            const uint64_t rem = pos < 64 ? stop >> pos : 0ull;
            if (rem == 0) {
                run += 64 - pos;
                rho -= 64;
                gam -= 64;
                break;
            }
            const int f = pos + __builtin_ctzll(rem);
            run += f - pos;
            if ((out >> f) & 1ull) {
                rho -= f;
                gam -= f;
                have = false;
                break;
            }
            const int op = (int)((hib >> f) & 1ull) * 2 + (int)((lob >> f) & 1ull);
            if (cnt >= p.L) return -1;
            push(op);
            if (op == OP_SUB) {  // the same diagonal goes on
                pos = f + 1;
                continue;
            }
            rho -= f + (op == OP_DEL ? 1 : 0);
            gam -= f + (op == OP_INS ? 1 : 0);
            break;
        }
    }
    const int left = rho >= 0 ? rho + 1 : gam + 1;  // rows or columns before the other's first
    if (cnt + left > p.L) return -1;
    for (int i = 0; i < left; ++i) push(rho >= 0 ? OP_DEL : OP_INS);
    if (cnt & 63) tok[(cnt & ~63) + lane] = (uint32_t)tokv;
    return cnt;
}

// The least key of a group of GL lanes (8 or 16), in every lane of it: lanes
// paired by DPP (the other of two, of two twos, the mirrored half row and row).
template <int GL>
__device__ __forceinline__ uint32_t group_min(uint32_t k) {
    k = min(k, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)k, 0xB1, 0xF, 0xF, true));   // quad_perm 1,0,3,2
    k = min(k, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)k, 0x4E, 0xF, 0xF, true));   // quad_perm 2,3,0,1
    k = min(k, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)k, 0x141, 0xF, 0xF, true));  // row_half_mirror
    if constexpr (GL == 16) k = min(k, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)k, 0x140, 0xF, 0xF, true));  // row_mirror
    return k;
}

// The path of the lane's pair as tokens (run << 2 | op), last op first, at tok.
// Returns the edits (-1: more than p.L) and in `run` the matches before the
// first op.
// A step: each lane looks at RL/GL cells of the path's diagonal and makes a key of
// the first that is an op or outside the tiles (steps back << 2 | op, op 0:
// outside); the group's least key is the next event.
template <int GL>
__device__ __forceinline__ int bp_walk(const BpPair& p, bool mine, const BpSegs& sg, const uint2* rec, uint32_t* tok,
                                       uint2* tiles, int& run, int lane) {
    typedef TraceShape<GL> T;
    static_assert(GL <= 16, "a group's tiles are one 16-bit mask");
    const int gl = lane & (GL - 1), g0 = lane & ~(GL - 1);
    int rho = p.plen - 1, gam = p.tlen - 1;  // the cell's row and column, from 0
    int cnt = 0;
    bool lost = p.L < 0;
    run = 0;
    uint2* const my = tiles + lane * TILE_WORDS;
    for (;;) {
        bool go = mine && !lost && rho >= 0 && gam >= 0;
        if (!__builtin_amdgcn_ballot_w64(go)) break;
        // tiles: words base, base + 1 (relative to the block) of blocks j0,
        // j0 - 1, ..
        const int j0 = gam >> 5;
        const int base = (rho - gam) >> 5;
        const int J = j0 - gl / T::TW;
        int S, w, at;
        bp_segment_of(sg, J, S, w, at);
        const int idx = base + gl % T::TW - S;  // word of the band
        // (a word above row 0 is outside: the path ends there)
        const bool have = go && J >= 0 && idx >= 0 && idx < GL * w && J + S + idx >= 0;
        const uint32_t tm = (uint32_t)group_bits<GL>(__builtin_amdgcn_ballot_w64(have), lane);
        group_sync<1>();
        if (have) bp_tile(p, rec, J, idx, S, w, at, g0, my, tile_swizzle(lane));
        group_sync<1>();
        // the lane's first cell, in columns left of the tiles' last column (G)
        // and rows below their first row (R)
        int G = 32 * j0 + 31 - gam + gl, R = rho - 32 * (j0 + base) - gl;
        const int G0 = G, R0 = R;
        bool fresh = true;
        while (__builtin_amdgcn_ballot_w64(go)) {
            uint32_t key = ~0u;
#pragma unroll
            for (int c = T::RL - GL; c >= 0; c -= GL) {
                const int q = (G + c) >> 5, u = ((R - c) >> 5) + q, t = q * T::TW + u;
                const bool in = (unsigned)u < (unsigned)T::TW && ((tm >> (t & 31)) & 1u);
                const uint2 cc = tiles[in ? (g0 + t) * TILE_WORDS + ((~(G + c) & 31) ^ tile_swizzle(g0 + t)) : 0];
                const uint32_t b = (uint32_t)(R - c) & 31u;
                const uint32_t op = in ? ((cc.x >> b) & 1u) << 1 | ((cc.y >> b) & 1u) : 0u;
                if (!in || op) key = (uint32_t)(gl + c) << 2 | op;
            }
            key = group_min<GL>(key);
            const bool event = key != ~0u;
            const int f = event ? (int)(key >> 2) : T::RL;
            const uint32_t op = key & 3u;
            const bool edit = event && op != 0u;
            if (go) {
                // on to new tiles at a cell outside these, unless it is the
                // first: then the path left the band, with more than L edits
                lost = event && !edit && fresh && f == 0;
                go = !event || edit;
                run += f;
                if (edit) {
                    if (gl == 0) tok[cnt] = (uint32_t)run << 2 | op;
                    ++cnt;
                    run = 0;
                }
                G += f + (edit && op != OP_DEL);
                R -= f + (edit && op != OP_INS);
                if (cnt > p.L) {
                    lost = true;
                    go = false;
                }
            }
            fresh = false;
        }
        gam -= G - G0;
        rho += R - R0;
    }
    if (!mine || lost) return -1;
    // rows or columns before the other's first
    const int left = rho >= 0 ? rho + 1 : gam + 1;
    if (cnt + left > p.L) return -1;
    const uint32_t op = rho >= 0 ? OP_DEL : OP_INS;
    for (int i = gl; i < left; i += GL) tok[cnt + i] = i == 0 ? (uint32_t)run << 2 | op : op;
    if (left > 0) run = 0;
    return cnt + left;
}

// The CIGAR stream of a pair from its tokens, by the whole wave, and its result
// (cnt edits, -1: deferred; run: the matches before the first op).
__device__ __forceinline__ void bp_emit(const BpArgs& a, uint32_t pidx, int cnt, int run, const uint32_t* tok, int lane) {
    ewfa_result_t* res = a.results + pidx;
    if (cnt < 0) {
        if (lane == 0) {
            a.defer_list[atomicAdd(a.defer_count, 1u)] = pidx;
            res->status = PAIR_DEFERRED;
        }
        return;
    }
    const uint64_t coff = a.pairs[pidx].cigar_off;
    const uint32_t cap = a.pairs[pidx].cigar_cap;
    if ((coff & 3u) || (cap & 3u)) {
        if (lane == 0) *res = ewfa_result_t{cnt, 0, EWFA_PAIR_BADARG, 0};
        return;
    }
    // step s's run and op from tokens cnt - s and cnt - 1 - s
    WaveStream w{a.cigars + coff, cap, 0u};
    for (int s0 = 0; s0 < cnt; s0 += 64) {
        const int s = s0 + lane;
        const bool act = s < cnt;
        const int op = act ? (int)(tok[cnt - 1 - s] & 3u) : 0;
        w.put(act, !act ? 0 : s == 0 ? run : (int)(tok[cnt - s] >> 2), op);
    }
    w.finish(cnt ? (int)(tok[0] >> 2) : run, lane);
    if (lane == 0)
        *res = ewfa_result_t{cnt, (int32_t)w.len, w.len > cap ? EWFA_PAIR_OVERFLOW : EWFA_PAIR_OK, 0};
}

// One wave's pairs: list[first ..] up to 64/GL of them, below `end`, of bands of
// N words.
template <int GL>
__device__ __forceinline__ void bp_item(const BpArgs& a, uint32_t first, uint32_t end, int N, uint2* rec, uint32_t* tok,
                                        uint2* tiles, int lane) {
    const uint32_t g = (uint32_t)(lane / GL);
    // lanes of groups past the list's end repeat its last pair, unwalked
    const uint32_t pidx = a.list[min(first + g, end - 1u)];
    const ewfa_pair_t pr = a.pairs[pidx];
    const int W = (N + GL - 1) / GL;
    const BpPair p = bp_load(a, pidx, pr, GL * W);
    int nblk = 0;
#pragma unroll
    for (int q = 0; q < 64 / GL; ++q) nblk = max(nblk, (int)__builtin_amdgcn_readlane(p.nwt, q * GL));
    BpSegs sg;
    bp_forward<GL>(p, W, nblk, rec, sg, reinterpret_cast<uint32_t*>(tiles), lane);
    __threadfence_block();  // the records are read back by other lanes
    int run = 0, cnt = 0;
    if constexpr (GL < 32) cnt = bp_walk<GL>(p, first + g < end, sg, rec, tok + g * bp_tok_stride(GL), tiles, run, lane);
    for (uint32_t q = 0; q < 64u / GL && first + q < end; ++q) {
        const int src = (int)q * GL;
        const uint32_t mine = (uint32_t)__builtin_amdgcn_readlane((int)pidx, src);
        uint32_t* const t = tok + q * bp_tok_stride(GL);
        if constexpr (GL < 32) {
            __threadfence_block();  // the tokens are read back by other lanes
            bp_emit(a, mine, __builtin_amdgcn_readlane(cnt, src), __builtin_amdgcn_readlane(run, src), t, lane);
        } else {
            const ewfa_pair_t pg = a.pairs[mine];
            const BpPair pu = bp_load(a, mine, pg, GL * W);
            BpSegs su = sg;
#pragma unroll
            for (int k = 0; k < 4; ++k) su.S[k] = __builtin_amdgcn_readlane(sg.S[k], src);
            const int c = bp_walk_wave<GL>(pu, su, src, rec, t, tiles, run, lane);
            __threadfence_block();
            bp_emit(a, mine, c, run, t, lane);
        }
    }
}

}  // namespace

// Persistent, one wave per block.  The list holds the pairs class by class,
// widest band first (BP_CLASSES classes from seg[c], seg[BP_CLASSES] the end),
// each by decreasing length; an item is the 64/GL pairs of a wave.  PART: the
// classes of 32 lanes and more (BP_WIDE), the others (BP_NARROW) or all.  Long
// reads take the first two one after the other, since the wide bands alone need
// half the LDS (four waves per SIMD instead of two and a half: 20,000 pairs of
// 10..50 kbp in 44.5 ms, 51.6 with one kernel for all); shorter pairs, of which
// few are wide, one kernel, whose narrow pairs hide the wide ones' long chains
// (15,001 pairs of 3..7 kbp at 8..15% edits: 3.5 ms, 4.9 apart).
template <int PART>
__global__ __launch_bounds__(64, PART == BP_WIDE ? 4 : 3) void bp_kernel(BpArgs a) {
    __shared__ uint2 tiles[TraceShape<PART == BP_WIDE ? 64 : 16>::TILES * TILE_WORDS];
    const int lane = threadIdx.x;
    if (a.seg[BP_CLASSES] == 0) return;
    uint8_t* slot = a.slots + (size_t)blockIdx.x * a.slot_bytes;
    uint32_t* tok = reinterpret_cast<uint32_t*>(slot);
    uint2* rec = reinterpret_cast<uint2*>(slot + a.tok_bytes);
    for (;;) {
        uint32_t item = wave_take(a.queue + (PART == BP_NARROW ? 1 : 0), 1u, lane);
        int c = 0, gl = 64;
        uint32_t lo = 0, hi = 0, per = 1;
        for (; c < BP_CLASSES; ++c) {
            gl = bp_group(c, a.spread);
            if (PART != BP_ALL && (gl >= 32) != (PART == BP_WIDE)) continue;
            lo = a.seg[c];
            hi = a.seg[c + 1];
            per = 64u / (uint32_t)gl;
            const uint32_t items = (hi - lo + per - 1u) / per;
            if (item < items) break;
            item -= items;
        }
        if (c == BP_CLASSES) break;
        const uint32_t first = lo + item * per;
        const int N = bp_words(c);
        if (PART != BP_NARROW && gl == 64) bp_item<64>(a, first, hi, N, rec, tok, tiles, lane);
        else if (PART != BP_NARROW && gl == 32) bp_item<32>(a, first, hi, N, rec, tok, tiles, lane);
        else if (PART != BP_WIDE && gl == 16) bp_item<16>(a, first, hi, N, rec, tok, tiles, lane);
        else if (PART != BP_WIDE) bp_item<8>(a, first, hi, N, rec, tok, tiles, lane);
        group_sync<1>();
    }
}

// Wave instructions of a wavefront search of d levels: weights fitted to calls, of
// the two-wave passes (500,000 pairs of 100..10,000 bp at 1..10% edits took 25.1,
// 20.6, 20.1 and 20.7 ms with 0.22, 0.5, 1 and 2 per d * d) and of the eight-wave
// passes within distance bounds, whose levels cost much the same until they are
// wider than the block (10..20 kbp pairs 0.55 us each at 1..3% edits and 1.6 at
// 5..12%, 10..50 kbp pairs 9.2 at 10..15%).
__device__ __forceinline__ float wavefront_cost(float d, bool deep) {
    return d * (deep ? 750.0f + 0.2f * d : 100.0f + 0.6f * d);
}
// Microseconds a wave instruction takes of the whole chip (256 CUs at about
// 2.3 GHz), and a column of a pair from table to path.
constexpr float BP_INSTR_US = 1.7e-6f, BP_COLUMN_US = 0.13f;

// Sum and maximum over the wave, in every lane.
__device__ __forceinline__ float wave_add(float v) {
    for (int d = 32; d; d >>= 1) v += __shfl_xor(v, d);
    return v;
}

__device__ __forceinline__ float wave_most(float v) {
    for (int d = 32; d; d >>= 1) v = fmaxf(v, __shfl_xor(v, d));
    return v;
}

// ---- distance bounds ------------------------------------------------------------
// An upper bound on each pair's distance from a window of 64 diagonals that
// follows the path: the same table, one pair per lane, the window's vertical
// deltas in a 64-bit word that moves down a row a column (so only the diagonal
// term shifts).  Every 32 columns the window moves by up to BAND_MOVE rows
// towards the edge with the smaller value.  Rows that enter it count +1 a row
// from the ones it holds, so every value is that of a real alignment.
// One lane per pair costs a sixth of the wave per pair of bound_kernel (a level
// there keeps 64 lanes for some 5 cells that matter) but takes tlen columns of
// about 80 ns however few pairs there are: it is for large lists.

namespace {

constexpr int BAND_MOVE = 12;

struct LaneBand {
    uint64_t vp, vn;
    int sc;  // value of the row above the window's first
    int r0;  // the window's first row (from 0) at the next column
};

// One column over 32-bit halves (64-bit shifts and adds take several cycles a
// lane): p, q the window's pattern planes' halves, c0, c1 the text base's masks;
// returns the low half of the diagonal-delta-0 vector (bit 0: the first row).
__device__ __forceinline__ uint32_t band_column(uint32_t (&vp)[2], uint32_t (&vn)[2], const uint32_t (&p)[2],
                                                const uint32_t (&q)[2], uint32_t c0, uint32_t c1) {
    uint32_t xh[2], ph[2], mh[2], xv[2];
    unsigned c = 0;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const uint32_t eq = ~(p[h] ^ c0) & ~(q[h] ^ c1);
        xh[h] = (__builtin_addc(eq & vp[h], vp[h], c, &c) ^ vp[h]) | eq;
        ph[h] = vn[h] | ~(xh[h] | vp[h]);
        mh[h] = vp[h] & xh[h];
        xv[h] = eq | vn[h];
    }
    const uint32_t d0 = xh[0] | vn[0];
    const uint32_t x0 = __builtin_amdgcn_alignbit(xv[1], xv[0], 1), x1 = xv[1] >> 1;
    vp[0] = mh[0] | ~(x0 | ph[0]);
    vp[1] = mh[1] | ~(x1 | ph[1]);
    vn[0] = ph[0] & x0;
    vn[1] = ph[1] & x1;
    return d0;
}

__device__ __forceinline__ uint32_t sign_mask(uint32_t planes, int i) { return (uint32_t)((int)(planes << (31 - i)) >> 31); }

// The bound, and in `slope` the least growth of the window's middle value over
// SLOPE_BLOCKS column blocks (the edit rate while the window was on the path;
// unchanged when the text has fewer).
// SAMPLE: the edits of the text's first tlen bases against whatever part of the
// pattern suits them, the least value of the last column (that of row tlen counts
// the path's distance from the diagonal as edits: half as many again for pairs of
// 4.5% in runs), and in `slope` the same of the first half of them.
constexpr int SLOPE_BLOCKS = 32;

template <bool SAMPLE = false>
__device__ uint32_t lane_bound(const uint64_t* gp, const uint64_t* gt, int plen, int tlen, int& slope) {
    const int nwp = (plen + 31) >> 5;
    int mid0 = 0;
    LaneBand b{~0ull << 32, ~0ull >> 32, 32, -32};
    uint32_t a[4], c[4];  // pattern planes from row r0 & ~31
    const auto load = [&]() {
        const int w = b.r0 >> 5;
#pragma unroll
        for (int x = 0; x < 4; ++x) planes_of(gp[min(max(w + x, 0), nwp)], a[x], c[x]);
        // ... moved so that bit 0 is row r0: 96 rows
        const uint32_t sh = (uint32_t)b.r0 & 31u;
#pragma unroll
        for (int x = 0; x < 3; ++x) {
            a[x] = __builtin_amdgcn_alignbit(a[x + 1], a[x], sh);
            c[x] = __builtin_amdgcn_alignbit(c[x + 1], c[x], sh);
        }
    };
    const auto column = [&](uint32_t (&vp)[2], uint32_t (&vn)[2], uint32_t t0, uint32_t t1, int i) -> uint32_t {
        const uint32_t p[2] = {__builtin_amdgcn_alignbit(a[1], a[0], (uint32_t)i), __builtin_amdgcn_alignbit(a[2], a[1], (uint32_t)i)};
        const uint32_t q[2] = {__builtin_amdgcn_alignbit(c[1], c[0], (uint32_t)i), __builtin_amdgcn_alignbit(c[2], c[1], (uint32_t)i)};
        return band_column(vp, vn, p, q, sign_mask(t0, i), sign_mask(t1, i));
    };
    // least value of the column over the pattern's rows
    const auto least = [&]() -> int {
        int v = b.sc, m = v;
        const int rows = min(plen - b.r0, 64);
        for (int i = 0; i < rows; ++i) {
            v += (int)((b.vp >> i) & 1u) - (int)((b.vn >> i) & 1u);
            m = min(m, v);
        }
        return m;
    };
    const int full = tlen >> 5;
    for (int j = 0; j < full; ++j) {
        if (SAMPLE && j == full / 2) slope = least();
        uint32_t t0, t1;
        load();
        planes_of(gt[j], t0, t1);
        uint32_t z = 0;
        uint32_t vp[2] = {(uint32_t)b.vp, (uint32_t)(b.vp >> 32)}, vn[2] = {(uint32_t)b.vn, (uint32_t)(b.vn >> 32)};
#pragma unroll
        for (int i = 0; i < 32; ++i) z = __builtin_amdgcn_alignbit(column(vp, vn, t0, t1, i), z, 1);
        b.vp = (uint64_t)vp[1] << 32 | vp[0];
        b.vn = (uint64_t)vn[1] << 32 | vn[0];
        b.sc += 32 - __popc(z);
        b.r0 += 32;
        // bottom edge's value less the top edge's, halved: rows to move up
        const int diff = __popcll(b.vp) - __popcll(b.vn);
        const int up = min(max(diff / 2, -BAND_MOVE), BAND_MOVE);
        if (up > 0) {
            b.vp <<= up;
            b.vn = (b.vn << up) | ((1ull << up) - 1ull);
            b.sc += up;
        } else if (up < 0) {
            const uint64_t m = (1ull << -up) - 1ull;
            b.sc += __popcll(b.vp & m) - __popcll(b.vn & m);
            b.vp = (b.vp >> -up) | ~(~0ull >> -up);
            b.vn >>= -up;
        }
        b.r0 -= up;
        if ((j & (SLOPE_BLOCKS - 1)) == SLOPE_BLOCKS - 1) {
            const int mid = b.sc + __popc((uint32_t)b.vp) - __popc((uint32_t)b.vn);
            slope = min(slope, mid - mid0);
            mid0 = mid;
        }
    }
    const int rest = tlen & 31;
    if (rest) {
        uint32_t t0, t1;
        load();
        planes_of(gt[full], t0, t1);
        uint32_t vp[2] = {(uint32_t)b.vp, (uint32_t)(b.vp >> 32)}, vn[2] = {(uint32_t)b.vn, (uint32_t)(b.vn >> 32)};
        for (int i = 0; i < rest; ++i) b.sc += 1 - (int)(column(vp, vn, t0, t1, i) & 1u);
        b.vp = (uint64_t)vp[1] << 32 | vp[0];
        b.vn = (uint64_t)vn[1] << 32 | vn[0];
        b.r0 += rest;
    }
    if constexpr (SAMPLE) return (uint32_t)least();
    // row plen - 1 of the last column
    const int idx = plen - b.r0;
    if (idx <= 0) return (uint32_t)(b.sc - idx);
    const uint64_t m = idx >= 64 ? ~0ull : (1ull << idx) - 1ull;
    return (uint32_t)(b.sc + __popcll(b.vp & m) - __popcll(b.vn & m) + max(idx - 64, 0));
}

}  // namespace

// Whether a list takes the bit-parallel way at all, from a sample: 256 of its
// pairs, a lane each, and the edits in the first PROBE_BASES of each (35 us).  The
// wavefront's time is the longer of its work and its longest pair's levels and three
// quarters of the other, and the levels once more and 2 us each for pairs beyond its
// budget; the bit-parallel one its work and its longest pair's columns and levels.
// Over 146 drawn lists of one bucket (1,030..60,000 pairs of 1.3..10.4 kbp at 0.2..15%
// edits) the median of the time by the estimate is 1.00 and 0.99, and of 210 lists 7
// went a way more than 6% behind the other.  The ways of 35,000 pairs of 5 kbp at 4%
// take 2.73 ms (wavefront) and 3.23, 2,500 of 4.3..8.7 kbp at 3..6% in runs
// 0.86 and 2.36; the other way round 35,000 of 5 kbp at 9% 7.32 and 3.71.
constexpr int PROBE_BASES = 256;
constexpr int PROBE_PAIRS = 256;
constexpr float FEW_LEVELS = 512.0f;

__global__ __launch_bounds__(PROBE_PAIRS) void bp_probe_kernel(BpArgs a, const uint32_t* list, const uint32_t* count_ptr,
                                                               uint32_t count, int budget, BpBeside beside,
                                                               uint32_t* flag) {
    const uint32_t n = count_ptr ? *count_ptr : count;
    if (n == 0) return;
    __shared__ float part[PROBE_PAIRS / 64][5];
    // over the block, in every thread: the sums of the first `sums` values, the
    // greatest of the others
    const auto join = [&](auto& v, int sums) {
        constexpr int N = (int)(sizeof v / sizeof v[0]);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < N; ++i) {
            v[i] = i < sums ? wave_add(v[i]) : wave_most(v[i]);
            if ((threadIdx.x & 63u) == 0u) part[threadIdx.x >> 6][i] = v[i];
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < N; ++i) {
            v[i] = part[0][i];
            for (int w = 1; w < PROBE_PAIRS / 64; ++w) v[i] = i < sums ? v[i] + part[w][i] : fmaxf(v[i], part[w][i]);
        }
    };
    const uint32_t item = (uint32_t)(((uint64_t)n * (2u * threadIdx.x + 1u)) / (2u * PROBE_PAIRS));
    const uint32_t pidx = list ? list[item] : item;
    const ewfa_pair_t pr = a.pairs[pidx];
    float edits = 0.f, second = 0.f, bases = 0.f, columns = 0.f;
    if (pr.plen <= a.max_len && pr.tlen <= a.max_len && pr.tlen > 0u) {
        const int tl = min((int)pr.tlen, PROBE_BASES);
        int half = 0;
        edits = (float)lane_bound<true>(a.words + pr.pattern_off, a.words + pr.text_off, (int)pr.plen, tl, half);
        second = edits - (float)half;
        bases = (float)tl;
        columns = (float)pr.tlen;
    }
    // the list's rate from the samples' second halves, since an end that is free
    // to choose saves an edit or two, the first half's as the whole's
    float s1[3] = {bases, edits, second};
    join(s1, 3);
    const float all = fmaxf(s1[0], 1.f), sum = fmaxf(s1[1], 1.f), mean = 2.f * s1[2] / all;
    // the pairs' rates, drawn to their mean by what the two halves of a sample show
    // to be the sample's own variance (edits come in runs): each to the likeliest
    // rate, and for the share of pairs beyond the budget only until the variance is
    // that of the rates
    const float off = bases > 0.f ? edits * all / (bases * sum) - 1.f : 0.f;
    const float diff = bases > 0.f ? (2.f * second - edits) * all / (bases * sum) : 0.f;
    float s2[2] = {off * off, diff * diff};
    join(s2, 2);
    const float keep = s2[0] > s2[1] ? 1.f - s2[1] / s2[0] : 0.f;
    const float levels = mean * fminf(1.f + off * keep, 2.5f) * columns;
    const bool beyond = mean * fminf(1.f + off * sqrtf(keep), 2.5f) * columns > (float)budget;
    // wave instructions of both ways: a two-wave search with its staging and stream
    // (35,000 pairs of 1.5, 2.4, 3.5 and 5 kbp at 2, 4 and 9% edits within 10%, from 493
    // us at 1.5 kbp and 2% to 7,322 at 5 kbp and 9%), and bounds, table and path
    float s3[5] = {levels * (95.0f + 0.29f * levels) + 2.9f * columns, columns * 7.5f + 25.0f * levels,
                   beyond ? 1.f : 0.f, levels, columns};
    join(s3, 3);
    const float most = s3[3], longest = s3[4];
    // wave instructions a microsecond: 256 CUs at about 2.3 GHz
    const float share = (float)n / (float)PROBE_PAIRS, us = share / 590000.0f;
    const float wfa = s3[0] * us, bp = s3[1] * us, deferred = s3[2] >= 3.f ? s3[2] * share : 0.f;
    const float chain = most * (1.1f + 0.0005f * most) * (deferred > 0.f ? 2.0f : 1.0f);
    const float wave_us = 1.1f * (fmaxf(wfa, chain) + 0.75f * fminf(wfa, chain)) + 2.0f * deferred;
    // other buckets' passes of twice this one's bases fill what its columns' chains
    // leave idle (500,000 pairs of 100..10,000 bp at 1..10%: 15.6 ms with the 80,000 of
    // 1.2..2.5 kbp by the wavefront, 15.0 without)
    const float columns_us = 0.2f * longest + 0.5f * most;
    float others = 0.f;
    for (int b = 0; b < beside.nb; ++b)
        if (b != beside.self) others += (float)beside.counts[b] * (float)beside.len[b];
    const bool hidden = beside.nb > 1 && others >= 2.f * (float)n * (float)beside.len[beside.self];
    const float bits_us = fmaxf(bp, columns_us) + (hidden ? 0.25f : 1.0f) * fminf(bp, columns_us);
    if (threadIdx.x == 0) *flag = bits_us < wave_us ? 1u : 0u;
}

// Splits a list of few long pairs between two passes, by the same sample: all of
// it goes to the one without distance bounds (counts[0]) while the longest pair has
// about as many levels as its block has lanes, which the bound search doubles (a
// level costs no less for fewer diagonals), else to the one within them
// (counts[1]).  512 pairs of 10..25 kbp at 0.5..2% edits take 736 us without and 875
// with bounds, at 5..8% 3,498 and 2,955.
__global__ __launch_bounds__(64) void few_probe_kernel(const uint64_t* words, const ewfa_pair_t* pairs, uint32_t max_len,
                                                       const uint32_t* list, const uint32_t* count_ptr, uint32_t count,
                                                       uint32_t* counts) {
    const uint32_t n = count_ptr ? *count_ptr : count;
    bool near = true;
    if (n) {
        const uint32_t item = (uint32_t)(((uint64_t)n * (2u * threadIdx.x + 1u)) / 128u);
        const ewfa_pair_t pr = pairs[list ? list[item] : item];
        float edits = 0.f, bases = 0.f, columns = 0.f;
        if (pr.plen <= max_len && pr.tlen <= max_len && pr.tlen > 0u) {
            const int tl = min((int)pr.tlen, PROBE_BASES), pl = min((int)pr.plen, PROBE_BASES);
            int slope = 0;
            edits = (float)lane_bound(words + pr.pattern_off, words + pr.text_off, pl, tl, slope);
            bases = (float)tl;
            columns = (float)pr.tlen;
        }
        near = wave_add(edits) * wave_most(columns) < FEW_LEVELS * wave_add(bases);
    }
    if (threadIdx.x == 0) {
        counts[0] = near ? n : 0u;
        counts[1] = near ? 0u : n;
    }
}

__global__ __launch_bounds__(64, 4) void bp_bound_kernel(const uint64_t* words, const ewfa_pair_t* pairs, uint32_t max_len,
                                                         uint32_t* bound, uint32_t* guess, uint32_t least, const uint32_t* list,
                                                         const uint32_t* count_ptr, uint32_t count,
                                                         const uint32_t* flag) {
    if (flag && *flag == 0u) return;
    const uint32_t n = count_ptr ? *count_ptr : count;
    if (n < least) return;
    for (uint32_t item = blockIdx.x * 64u + threadIdx.x; item < n; item += gridDim.x * 64u) {
        const uint32_t pidx = list ? list[item] : item;
        const ewfa_pair_t pr = pairs[pidx];
        uint32_t u = BOUND_NONE, d = BOUND_NONE;
        if (pr.plen <= max_len && pr.tlen <= max_len) {
            int slope = 1 << 20;
            u = lane_bound(words + pr.pattern_off, words + pr.text_off, (int)pr.plen, (int)pr.tlen, slope);
            // a guess at the distance for when the window lost the path
            if (slope < (1 << 20))
                d = (uint32_t)((float)max(slope, 0) * 1.25f * (float)pr.tlen / (32.0f * SLOPE_BLOCKS)) + 64u;
        }
        bound[pidx] = u;
        guess[pidx] = min(u, d);
    }
}

hipError_t launch_bp_bound(const BpArgs& a, uint32_t* bound, const uint32_t* list, const uint32_t* count_ptr,
                           uint32_t count, uint32_t max_grid, hipStream_t stream) {
    if (count == 0) return hipSuccess;
    const uint32_t blocks = (count + 63u) / 64u;
    hipLaunchKernelGGL(bp_bound_kernel, dim3(blocks < max_grid ? blocks : max_grid), dim3(64), 0, stream, a.words,
                       a.pairs, a.max_len, bound, a.guess, a.lane_min, list, count_ptr, count, a.flag);
    return hipGetLastError();
}

hipError_t launch_few_probe(const uint64_t* words, const ewfa_pair_t* pairs, uint32_t max_len, const uint32_t* list,
                            const uint32_t* count_ptr, uint32_t count, uint32_t* counts, hipStream_t stream) {
    hipLaunchKernelGGL(few_probe_kernel, dim3(1), dim3(64), 0, stream, words, pairs, max_len, list, count_ptr, count,
                       counts);
    return hipGetLastError();
}

hipError_t launch_bp_probe(const BpArgs& a, const uint32_t* list, const uint32_t* count_ptr, uint32_t count,
                           int budget, const BpBeside& beside, uint32_t* flag, hipStream_t stream) {
    hipLaunchKernelGGL(bp_probe_kernel, dim3(1), dim3(PROBE_PAIRS), 0, stream, a, list, count_ptr, count, budget, beside, flag);
    return hipGetLastError();
}

// ---- which pairs come here -----------------------------------------------------

namespace {

constexpr float LOST_RATE = 0.15f;

// What a pair costs each way: wave instructions of the chip's work, and the us its
// own chain takes: its levels (about 1.1 us and half a ns a diagonal each, its
// stream included; twice where the pass's budget of levels defers it), or its
// columns.
struct BpCost {
    int c;  // class: the narrowest band that holds every path within the bound
            // (BP_CLASSES: no bound, the pair is the wavefront's)
    float wave, bits, wave_us, bits_us;
    float edits, bases;
    float lost_us;  // a pair without a bound: its levels if it has LOST_RATE edits a base
};

__device__ __forceinline__ float bp_levels_us(const BpArgs& a, float d) {
    return d * (1.1f + 0.0005f * d) * (d > (float)a.budget ? 2.0f : 1.0f);
}

// A bound beyond the widest band, or above a fifth of the text, mostly comes of a
// search whose window lost the path at a long gap: it then says nothing of the
// distance.  The guess from the part before the gap then gives the costs, and a
// bound beyond the widest band takes that band, where the distance most likely
// lies (if not the pair is deferred); without a guess such pairs stay with the
// wavefront.
__device__ __forceinline__ BpCost bp_cost(const BpArgs& a, uint32_t pidx, uint32_t n) {
    BpCost k{BP_CLASSES, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    const auto levels_us = [&](float d) { return bp_levels_us(a, d); };
    const ewfa_pair_t pr = a.pairs[pidx];
    uint32_t u = a.bound[pidx];
    if (pr.plen > a.max_len || pr.tlen > a.max_len || pr.tlen == 0u || pr.plen == 0u) return k;
    if (u == BOUND_NONE) {
        k.lost_us = levels_us(LOST_RATE * (float)pr.tlen);
        return k;
    }
    const int tk = (int)pr.tlen - (int)pr.plen;
    int S, c = BP_CLASSES - 1;
    while (c > 0 && bp_band(bp_words(c), tk, S) < (int)u) --c;
    const int L = bp_band(bp_words(c), tk, S);
    if (L < (int)u || u > pr.tlen / 5u + 64u) {
        k.lost_us = levels_us(LOST_RATE * (float)pr.tlen);
        if (!a.guess || n < a.lane_min || L < 0) return k;
        u = a.guess[pidx];
    }
    const float d = (float)u, cols = (float)pr.tlen;
    k.c = c;
    k.wave = wavefront_cost(d, a.deep);
    k.bits = cols * (bp_column_cost(c) + 2.0f) + 25.0f * d;
    // (few pairs have lost their path, and their guesses are rough: they are no
    // measure of the list's chains)
    k.wave_us = k.lost_us > 0.f ? 0.f : levels_us(d);
    k.bits_us = cols * BP_COLUMN_US;
    k.edits = d;
    k.bases = cols;
    return k;
}

// The list's way, from its pairs' costs together: every pair by the wavefront
// (0), each the way with less work (1), or every pair that has a class by the
// bit-parallel kernel (2).  A way's time is its work and its longest chain, of
// which they hide about half (1,500, 5,000 and 15,000 pairs of 10..20 kbp at
// 1..3% edits: 1.8, 3.4 and 9.0 ms by the wavefront, 3.0, 3.4 and 6.4
// bit-parallel); the two ways of one list run one after the other.  A pair without
// a bound starts first in a wavefront pass, beside the others; without a class it
// is the wavefront's in any case, after the bit-parallel kernels (3,462 pairs of
// 12..25 kbp, 61 of them such: 14.0 ms by the wavefront, 15.4 both ways).
__device__ __forceinline__ int bp_way(const BpWeigh& w, const BpArgs& a) {
    auto time = [](uint64_t work, uint32_t chain) {
        const float t = (float)work * BP_INSTR_US, l = (float)chain;
        return fmaxf(t, l) + 0.5f * fminf(t, l);
    };
    // (a loose bound is no distance: no chain of more than 2.5 times the mean rate;
    // in a deep bucket, whose lists no sample has passed, of 1.5 times, that of a pair
    // without a bound of 2.5, and a tenth in the wavefront's favour: a gap that loses
    // the path there triples a bound, and widens the classes.  1,450 pairs of 4.8..24
    // kbp at 3.6..6% in runs took 8.6 ms bit-parallel and take 3.6)
    const float longest = (float)w.edits / (float)max(w.bases, (uint64_t)1) * (float)w.bits_us / BP_COLUMN_US;
    const float most = bp_levels_us(a, (a.deep ? 1.5f : 2.5f) * longest);
    const float lost = a.deep ? bp_levels_us(a, 2.5f * longest) : 1e9f;
    const float rest_us = fminf((float)w.rest_us, lost);
    // (wide and narrow classes of a deep bucket run one after the other)
    const uint32_t twice = a.deep && w.wide_us ? w.wide_us : 0u;
    const float t0 = fmaxf(time(w.wave, min(w.wave_us, (uint32_t)most)), fmaxf(fminf((float)w.lost_us, lost), rest_us));
    const float t1 = time(w.split_bits, w.split_bits_us + twice) +
                     time(w.split_wave, min(w.split_wave_us, (uint32_t)most)) + rest_us;
    const float t2 = time(w.bits, w.bits_us + twice) + rest_us;
    return (a.deep ? 0.9f : 1.0f) * t0 <= fminf(t1, t2) ? 0 : t1 <= t2 ? 1 : 2;
}

// Bin of a pair in the sort: its class, then its length, longest first.
__device__ __forceinline__ int bp_bin_of(const BpArgs& a, uint32_t pidx, int way, uint32_t n) {
    int c = BP_CLASSES;
    if (way) {
        const BpCost k = bp_cost(a, pidx, n);
        if (way == 2 || k.bits <= k.wave) c = k.c;
    }
    const uint32_t b = min((uint32_t)((uint64_t)a.pairs[pidx].tlen * BP_LEN_BINS / (a.max_len + 1u)), (uint32_t)BP_LEN_BINS - 1u);
    return c * BP_LEN_BINS + (int)(BP_LEN_BINS - 1u - b);
}

// The way of a list: what the sample said, else its pairs' sums.
__device__ __forceinline__ int bp_list_way(const BpArgs& a) {
    return a.flag && *a.flag == 0u ? 0 : bp_way(*a.weigh, a);
}

}  // namespace

// Adds up the costs of the list's pairs (a.weigh, zero at first).
__global__ __launch_bounds__(256) void bp_weigh_kernel(BpArgs a, const uint32_t* list, const uint32_t* count_ptr,
                                                       uint32_t count) {
    const uint32_t n = count_ptr ? *count_ptr : count;
    if (a.flag && *a.flag == 0u) return;
    float sum[6] = {}, most[7] = {};
    for (uint32_t at = blockIdx.x * 256u + threadIdx.x; at < n; at += gridDim.x * 256u) {
        const BpCost k = bp_cost(a, list ? list[at] : at, n);
        const bool bits = k.bits <= k.wave;
        if (k.c == BP_CLASSES) {
            most[5] = fmaxf(most[5], k.lost_us);
            continue;
        }
        sum[0] += k.wave;
        sum[1] += k.bits;
        sum[2] += bits ? 0.f : k.wave;
        sum[3] += bits ? k.bits : 0.f;
        most[0] = fmaxf(most[0], k.wave_us);
        most[1] = fmaxf(most[1], k.bits_us);
        most[2] = fmaxf(most[2], bits ? 0.f : k.wave_us);
        most[3] = fmaxf(most[3], bits ? k.bits_us : 0.f);
        sum[4] += k.edits;
        sum[5] += k.bases;
        most[4] = fmaxf(most[4], k.lost_us);
        most[6] = fmaxf(most[6], bp_group(k.c, a.spread) >= 32 ? k.bits_us : 0.f);
    }
    // one wave of the block adds for all (each wave for itself took 0.1 to 0.4 ms of
    // adds to one line for 80,000 pairs)
    constexpr int SUMS = 6, ALL = SUMS + 7;
    __shared__ float part[4][ALL];
    const int wv = threadIdx.x >> 6;
#pragma unroll
    for (int i = 0; i < ALL; ++i) {
        const float v = i < SUMS ? wave_add(sum[i]) : wave_most(most[i - SUMS]);
        if ((threadIdx.x & 63u) == 0u) part[wv][i] = v;
    }
    __syncthreads();
    const int i = threadIdx.x;
    if (i < SUMS) {
        const float v = part[0][i] + part[1][i] + part[2][i] + part[3][i];
        if (v > 0.f) atomicAdd((unsigned long long*)(&a.weigh->wave + i), (unsigned long long)v);
    } else if (i < ALL) {
        const float m = fmaxf(fmaxf(part[0][i], part[1][i]), fmaxf(part[2][i], part[3][i]));
        if (m > 0.f) atomicMax(&a.weigh->wave_us + (i - SUMS), (uint32_t)m);
    }
}

// Counts the list's pairs per bin.
__global__ __launch_bounds__(256) void bp_count_kernel(BpArgs a, const uint32_t* list, const uint32_t* count_ptr,
                                                       uint32_t count) {
    __shared__ uint32_t h[BP_BINS];
    const uint32_t n = count_ptr ? *count_ptr : count;
    const uint32_t base = blockIdx.x * 256u;
    if (base >= n) return;
    const int way = bp_list_way(a);
    for (int i = threadIdx.x; i < BP_BINS; i += 256) h[i] = 0u;
    __syncthreads();
    const uint32_t at = base + threadIdx.x;
    if (at < n) {
        const uint32_t pidx = list ? list[at] : at;
        atomicAdd(&h[bp_bin_of(a, pidx, way, n)], 1u);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < BP_BINS; i += 256)
        if (h[i]) atomicAdd(a.bins + i, h[i]);
}

// Places them: the bit-parallel classes in a.list in bin order, the others in
// a.rest; the classes' ends in a.seg, the count of the others in a.rest_count.
__global__ __launch_bounds__(256) void bp_place_kernel(BpArgs a, const uint32_t* list, const uint32_t* count_ptr,
                                                       uint32_t count) {
    __shared__ uint32_t at[BP_BINS];  // the bins' first places
    __shared__ uint32_t h[BP_BINS], mine[BP_BINS];
    const uint32_t n = count_ptr ? *count_ptr : count;
    const uint32_t base = blockIdx.x * 256u;
    if (base >= n && blockIdx.x) return;
    const int way = bp_list_way(a);
    constexpr int FIRST_REST = BP_CLASSES * BP_LEN_BINS, BINS = 8;
    for (int i = threadIdx.x; i < BP_BINS; i += 256) h[i] = 0u;
    if (threadIdx.x < 64) {
        // running sums of the classes' bins, and of the rest's, BINS bins a lane
        constexpr int LANES = FIRST_REST / BINS, REST = BP_BINS - FIRST_REST;
        static_assert(FIRST_REST % BINS == 0 && LANES + (REST + BINS - 1) / BINS <= 64, "a wave holds the bins");
        const int lane = threadIdx.x;
        const int from = lane * BINS;
        uint32_t c[BINS], sum = 0;
#pragma unroll
        for (int i = 0; i < BINS; ++i) {
            c[i] = from + i < BP_BINS ? a.bins[from + i] : 0u;
            sum += c[i];
        }
        const uint32_t upto = (uint32_t)wave_incl_scan_i32((int)sum);
        const uint32_t classes = (uint32_t)__builtin_amdgcn_readlane((int)upto, LANES - 1);
        const uint32_t all = (uint32_t)__builtin_amdgcn_readlane((int)upto, 63);
        uint32_t run = upto - sum - (lane >= LANES ? classes : 0u);
#pragma unroll
        for (int i = 0; i < BINS; ++i) {
            const int bin = from + i;
            if (bin < BP_BINS) at[bin] = run;
            if (blockIdx.x == 0 && bin < FIRST_REST && bin % BP_LEN_BINS == 0) a.seg[bin / BP_LEN_BINS] = run;
            run += c[i];
        }
        if (blockIdx.x == 0 && lane == 0) {
            a.seg[BP_CLASSES] = classes;
            *a.rest_count = all - classes;
        }
    }
    __syncthreads();
    const uint32_t item = base + threadIdx.x;
    int b = -1;
    uint32_t pidx = 0, local = 0;
    if (item < n) {
        pidx = list ? list[item] : item;
        b = bp_bin_of(a, pidx, way, n);
        local = atomicAdd(&h[b], 1u);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < BP_BINS; i += 256)
        if (h[i]) mine[i] = atomicAdd(a.cursors + i, h[i]);
    __syncthreads();
    if (b >= 0) (b < FIRST_REST ? a.list_out : a.rest)[at[b] + mine[b] + local] = pidx;
}

hipError_t launch_bp_sort(const BpArgs& a, const uint32_t* list, const uint32_t* count_ptr, uint32_t count,
                          hipStream_t stream) {
    if (count == 0) return hipSuccess;
    const uint32_t blocks = (count + 255u) / 256u;
    hipLaunchKernelGGL(bp_weigh_kernel, dim3(blocks < 128u ? blocks : 128u), dim3(256), 0, stream, a, list, count_ptr, count);
    hipLaunchKernelGGL(bp_count_kernel, dim3(blocks), dim3(256), 0, stream, a, list, count_ptr, count);
    hipLaunchKernelGGL(bp_place_kernel, dim3(blocks), dim3(256), 0, stream, a, list, count_ptr, count);
    return hipGetLastError();
}

hipError_t launch_bp(const BpArgs& a, int part, uint32_t grid, hipStream_t stream) {
    if (grid == 0) return hipSuccess;
    switch (part) {
        case BP_WIDE: hipLaunchKernelGGL(bp_kernel<BP_WIDE>, dim3(grid), dim3(64), 0, stream, a); break;
        case BP_NARROW: hipLaunchKernelGGL(bp_kernel<BP_NARROW>, dim3(grid), dim3(64), 0, stream, a); break;
        default: hipLaunchKernelGGL(bp_kernel<BP_ALL>, dim3(grid), dim3(64), 0, stream, a); break;
    }
    return hipGetLastError();
}

int bp_blocks_per_cu(int part) {
    int blocks = 0;
    const void* f = part == BP_WIDE     ? reinterpret_cast<const void*>(&bp_kernel<BP_WIDE>)
                    : part == BP_NARROW ? reinterpret_cast<const void*>(&bp_kernel<BP_NARROW>)
                                        : reinterpret_cast<const void*>(&bp_kernel<BP_ALL>);
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, f, 64, 0) != hipSuccess) return 0;
    return blocks;
}

}  // namespace ewfa
