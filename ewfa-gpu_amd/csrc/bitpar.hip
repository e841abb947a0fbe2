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
    if constexpr (GL == 16) {  // row_shr:1
        return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xF, 0xF, true);
    } else {  // wave_shr:1
        const uint32_t y = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x138, 0xF, 0xF, true);
        if constexpr (GL == 32) return lane == 32 ? 0u : y;
        return y;
    }
}

// A lane's value from the lane after it in its group; a group's last lane
// gets `bottom`.
template <int GL>
__device__ __forceinline__ uint32_t from_below(uint32_t x, uint32_t bottom, int lane) {
    if constexpr (GL == 16) {  // row_shl:1
        return (uint32_t)__builtin_amdgcn_update_dpp((int)bottom, (int)x, 0x101, 0xF, 0xF, false);
    } else {  // wave_shl:1
        const uint32_t y = (uint32_t)__builtin_amdgcn_update_dpp((int)bottom, (int)x, 0x130, 0xF, 0xF, false);
        if constexpr (GL == 32) return lane == 31 ? bottom : y;
        return y;
    }
}

struct BpPair {
    const uint64_t* gp;  // packed words
    const uint64_t* gt;
    int plen, tlen, nwp, nwt;
    int S, L;            // band: words j + S .. j + S + N - 1 at column block j
};

__device__ __forceinline__ BpPair bp_load(const BpArgs& a, const ewfa_pair_t& pr, int N) {
    BpPair p;
    p.gp = a.words + pr.pattern_off;
    p.gt = a.words + pr.text_off;
    p.plen = (int)pr.plen;
    p.tlen = (int)pr.tlen;
    p.nwp = (p.plen + 31) >> 5;
    p.nwt = (p.tlen + 31) >> 5;
    p.L = bp_band(N, p.tlen - p.plen, p.S);
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
// the horizontal deltas below the lane's last row (nhp: those that are not +1).
// 18 vector instructions at W = 1, 12 to 14 per word more.
template <int GL, int W>
__device__ __forceinline__ void bp_column(uint32_t (&Pv)[W], uint32_t (&Mv)[W], const uint32_t (&P0)[W],
                                          const uint32_t (&P1)[W], uint32_t c0, uint32_t c1, uint32_t& nhp,
                                          uint32_t& hm, int lane) {
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
    nhp = __builtin_amdgcn_alignbit(nhp, nPh[W - 1], 31);
    hm = __builtin_amdgcn_alignbit(hm, Mh[W - 1], 31);
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

// The table's deltas of 64/GL pairs (p: the lane's own), column block by column
// block of 32.  rec gets, per block, every lane's vertical deltas at its start
// (W uint2 of Pv, Mv) and the horizontal deltas below its last row over the
// block (a uint2, column i at bit 31 - i): 64 * (W + 1) uint2.
template <int GL, int W>
__device__ __forceinline__ void bp_forward(const BpPair& p, int nblk, uint2* rec, int lane) {
    constexpr int N = GL * W;
    const int gl = lane & (GL - 1);
    uint32_t Pv[W], Mv[W], P0[W], P1[W];
#pragma unroll
    for (int w = 0; w < W; ++w) {
        // rows above the first (negative words) count down to it, so that row
        // 0 holds h in every column whatever their bases
        const int A = p.S + gl * W + w;
        Pv[w] = A < 0 ? 0u : ~0u;
        Mv[w] = A < 0 ? ~0u : 0u;
        planes_of(p.gp[min(max(A, 0), p.nwp)], P0[w], P1[w]);
    }
    for (int jb = 0; jb < nblk; jb += GL) {
        // the next GL blocks' text planes and the pattern planes that enter
        // the band with them, one per lane
        uint32_t f0, f1, e0, e1;
        planes_of(p.gt[min(jb + gl, p.nwt)], f0, f1);
        planes_of(p.gp[min(max(jb + gl + p.S + N - 1, 0), p.nwp)], e0, e1);
        const int nx = min(GL, nblk - jb);
        for (int x = 0; x < nx; ++x) {
            uint32_t T0, T1, q0, q1;
            if constexpr (GL == 64) {
                T0 = (uint32_t)__builtin_amdgcn_readlane((int)f0, x);
                T1 = (uint32_t)__builtin_amdgcn_readlane((int)f1, x);
                q0 = (uint32_t)__builtin_amdgcn_readlane((int)e0, x);
                q1 = (uint32_t)__builtin_amdgcn_readlane((int)e1, x);
            } else {
                const int at = ((lane & ~(GL - 1)) + x) << 2;
                T0 = (uint32_t)__builtin_amdgcn_ds_bpermute(at, (int)f0);
                T1 = (uint32_t)__builtin_amdgcn_ds_bpermute(at, (int)f1);
                q0 = (uint32_t)__builtin_amdgcn_ds_bpermute(at, (int)e0);
                q1 = (uint32_t)__builtin_amdgcn_ds_bpermute(at, (int)e1);
            }
            if (jb + x > 0) {  // the band moves down a word
                const uint32_t nPv = from_below<GL>(Pv[0], ~0u, lane);
                const uint32_t nMv = from_below<GL>(Mv[0], 0u, lane);
                const uint32_t n0 = from_below<GL>(P0[0], q0, lane);
                const uint32_t n1 = from_below<GL>(P1[0], q1, lane);
#pragma unroll
                for (int w = 0; w + 1 < W; ++w) {
                    Pv[w] = Pv[w + 1];
                    Mv[w] = Mv[w + 1];
                    P0[w] = P0[w + 1];
                    P1[w] = P1[w + 1];
                }
                Pv[W - 1] = nPv;
                Mv[W - 1] = nMv;
                P0[W - 1] = n0;
                P1[W - 1] = n1;
            }
#pragma unroll
            for (int w = 0; w < W; ++w) rec[w * 64 + lane] = make_uint2(Pv[w], Mv[w]);
            uint32_t nhp = 0, hm = 0;
            for (int i8 = 0; i8 < 32; i8 += 8) {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const uint32_t c0 = (uint32_t)((int)(T0 << (31 - i)) >> 31);
                    const uint32_t c1 = (uint32_t)((int)(T1 << (31 - i)) >> 31);
                    bp_column<GL, W>(Pv, Mv, P0, P1, c0, c1, nhp, hm, lane);
                }
                T0 >>= 8;
                T1 >>= 8;
            }
            rec[W * 64 + lane] = make_uint2(~nhp, hm);
            rec += 64 * (W + 1);
        }
    }
}

// ---- traceback ---------------------------------------------------------------
// The path is walked back over tiles of 32 rows x 32 columns whose op codes are
// computed again from the recorded deltas, TRACE_TILES at a time, a lane each:
// TRACE_WORDS row words around the path's diagonal over TRACE_BLOCKS column
// blocks.  The codes (two bits a cell, equal to OP_*, 0 for a match) go to LDS,
// where the whole wave looks along the diagonal at once: lane i at the cell i
// steps back, so a match run of up to 64 bases and the op that ends it are one
// ballot.
constexpr int TRACE_WORDS = 4, TRACE_BLOCKS = 8, TRACE_TILES = TRACE_WORDS * TRACE_BLOCKS;
constexpr int TILE_STRIDE = 33;  // uint2 per tile: a column each, and one that spreads the banks

template <int W>
__device__ __forceinline__ void trace_tile(const BpPair& p, const uint2* rec, int lane0, int J, int l, int w,
                                           uint2* out) {
    const uint2* rj = rec + (size_t)J * (64 * (W + 1));
    uint32_t pv[W], mv[W], p0[W], p1[W], T0, T1;
#pragma unroll
    for (int x = 0; x < W; ++x) {
        const uint2 d = rj[x * 64 + lane0 + l];
        pv[x] = d.x;
        mv[x] = d.y;
        planes_of(p.gp[min(max(J + p.S + l * W + x, 0), p.nwp)], p0[x], p1[x]);
    }
    uint2 h = make_uint2(~0u, 0u);
    if (l > 0) h = rj[W * 64 + lane0 + l - 1];
    planes_of(p.gt[min(J, p.nwt)], T0, T1);
#pragma unroll 4
    for (int i = 0; i < 32; ++i) {
        const uint32_t c0 = (uint32_t)((int)(T0 << (31 - i)) >> 31);
        const uint32_t c1 = (uint32_t)((int)(T1 << (31 - i)) >> 31);
        uint32_t ip = (h.x >> (31 - i)) & 1u, im = (h.y >> (31 - i)) & 1u;
        uint32_t hi = 0, lo = 0;
#pragma unroll
        for (int x = 0; x < W; ++x) {
            const uint32_t E = ~(p0[x] ^ c0) & ~(p1[x] ^ c1);
            const uint32_t Xv = E | mv[x];
            const uint32_t Eq = E | im;
            const uint32_t Xh = (((Eq & pv[x]) + pv[x]) ^ pv[x]) | Eq;
            const uint32_t Ph = mv[x] | ~(Xh | pv[x]), Mh = pv[x] & Xh;
            const uint32_t D0 = Xh | mv[x];  // diagonal delta 0
            const uint32_t ps = (Ph << 1) | ip, ms = (Mh << 1) | im;
            ip = Ph >> 31;
            im = Mh >> 31;
            pv[x] = ms | ~(Xv | ps);
            mv[x] = ps & Xv;
            // DEL 3: vertical +1; else SUB 2: diagonal +1; else INS 1: horizontal +1
            const uint32_t h1 = pv[x] | ~D0;
            const uint32_t l1 = pv[x] | (Ph & ~h1);
            hi = x == w ? h1 : hi;
            lo = x == w ? l1 : lo;
        }
        out[i] = make_uint2(hi, lo);
    }
}

// Bytes of a run of r matches in the stream.
__device__ __forceinline__ int run_bytes(int r) { return (r + 126) / 127; }

// The path of pair `pidx` (records in lanes lane0 .. of rec) as tokens
// (run << 2 | op), last op first, then its CIGAR stream and result.
template <int GL, int W>
__device__ __forceinline__ void bp_finish(const BpArgs& a, uint32_t pidx, const ewfa_pair_t& pr, const BpPair& p,
                                          int lane0, const uint2* rec, uint32_t* tok, uint2* tiles, int lane) {
    constexpr int N = GL * W;
    ewfa_result_t* res = a.results + pidx;
    int rho = p.plen - 1, gam = p.tlen - 1;  // the cell's row and column, from 0
    int run = 0, cnt = 0, tokv = 0;
    bool lost = p.L < 0;
    const auto push = [&](int op) {
        tokv = writelane_i32(tokv, (run << 2) | op, cnt & 63);
        run = 0;
        ++cnt;
        if ((cnt & 63) == 0) tok[cnt - 64 + lane] = (uint32_t)tokv;
    };
    int j0 = 0, base = 0;
    bool have = false;
    while (rho >= 0 && gam >= 0 && !lost) {
        const bool fresh = !have;
        if (!have) {
            j0 = gam >> 5;
            base = (rho - gam - 32) >> 5;  // the path's diagonal in the middle words
            const int t = lane & (TRACE_TILES - 1);
            const int J = j0 - t / TRACE_WORDS;
            const int idx = base + t % TRACE_WORDS - p.S;  // word of the band
            group_sync<1>();
            if (lane < TRACE_TILES && J >= 0 && idx >= 0 && idx < N)
                trace_tile<W>(p, rec, lane0, J, idx / W, idx % W, tiles + t * TILE_STRIDE);
            group_sync<1>();
            have = true;
        }
        const int r = rho - lane, g = gam - lane;
        const int J = g >> 5, q = j0 - J, u = (r >> 5) - J - base;
        const bool in = r >= 0 && g >= 0 && q < TRACE_BLOCKS && (unsigned)u < (unsigned)TRACE_WORDS &&
                        (unsigned)(base + u - p.S) < (unsigned)N;
        const uint2 cc = tiles[in ? (q * TRACE_WORDS + u) * TILE_STRIDE + (g & 31) : 0];
        const uint64_t hib = __builtin_amdgcn_ballot_w64(in && ((cc.x >> (r & 31)) & 1u));
        const uint64_t lob = __builtin_amdgcn_ballot_w64(in && ((cc.y >> (r & 31)) & 1u));
        const uint64_t out = __builtin_amdgcn_ballot_w64(!in);
        const uint64_t stop = hib | lob | out;
        if (fresh && (out & 1ull)) {  // outside the band: no path within L edits
            lost = true;
            break;
        }
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
            if (cnt >= p.L) {
                lost = true;
                break;
            }
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
    if (lost || cnt + left > p.L) {
        if (lane == 0) {
            a.defer_list[atomicAdd(a.defer_count, 1u)] = pidx;
            res->status = PAIR_DEFERRED;
        }
        return;
    }
    if ((pr.cigar_off & 3u) || (pr.cigar_cap & 3u)) {
        if (lane == 0) *res = ewfa_result_t{cnt + left, 0, EWFA_PAIR_BADARG, 0};
        return;
    }
    for (int i = 0; i < left; ++i) push(rho >= 0 ? OP_DEL : OP_INS);
    if (cnt & 63) tok[(cnt & ~63) + lane] = (uint32_t)tokv;
    __threadfence_block();  // the tokens are read back by other lanes
    // the stream: step s's run and op from tokens cnt - s and cnt - 1 - s
    int8_t* out = a.cigars + pr.cigar_off;
    const uint32_t cap = pr.cigar_cap;
    uint32_t at0 = 0;
    const auto put_run = [&](uint32_t at, int rb) -> uint32_t {
        for (; rb >= 127; rb -= 127, ++at)
            if (at < cap) out[at] = (int8_t)-127;
        if (rb) {
            if (at < cap) out[at] = (int8_t)-rb;
            ++at;
        }
        return at;
    };
    for (int s0 = 0; s0 < cnt; s0 += 64) {
        const int s = s0 + lane;
        const bool act = s < cnt;
        const int op = act ? (int)(tok[cnt - 1 - s] & 3u) : 0;
        const int rb = !act ? 0 : s == 0 ? run : (int)(tok[cnt - s] >> 2);
        const int nb = act ? run_bytes(rb) + 1 : 0;
        const int incl = wave_incl_scan_i32(nb);
        if (act) {
            const uint32_t at = put_run(at0 + (uint32_t)(incl - nb), rb);
            if (at < cap) out[at] = (int8_t)(op == OP_DEL ? 'D' : op == OP_SUB ? 'X' : 'I');
        }
        at0 += (uint32_t)__builtin_amdgcn_readlane(incl, 63);
    }
    const int fin = cnt ? (int)(tok[0] >> 2) : run;
    const uint32_t len = at0 + (uint32_t)run_bytes(fin);
    if (lane == 0) {
        put_run(at0, fin);
        // the terminator: zeros to the end of its dword, inside the region
        const uint32_t end = min((len & ~3u) + 4u, cap);
        for (uint32_t i = len; i < end; ++i) out[i] = 0;
        *res = ewfa_result_t{cnt, (int32_t)len, len > cap ? EWFA_PAIR_OVERFLOW : EWFA_PAIR_OK, 0};
    }
}

template <int GL, int W>
__device__ __forceinline__ void bp_item(const BpArgs& a, const uint32_t* list, uint32_t first, uint32_t count,
                                        uint2* rec, uint32_t* tok, uint2* tiles, int lane) {
    constexpr int NG = 64 / GL;
    // lanes of groups past the list's end repeat its last pair
    const uint32_t mine = list[min(first + (uint32_t)(lane / GL), count - 1u)];
    const ewfa_pair_t pr = a.pairs[mine];
    const BpPair p = bp_load(a, pr, GL * W);
    int nblk = 0;
#pragma unroll
    for (int g = 0; g < NG; ++g) nblk = max(nblk, (int)__builtin_amdgcn_readlane(p.nwt, g * GL));
    bp_forward<GL, W>(p, nblk, rec, lane);
    __threadfence_block();  // the records are read back by other lanes
    for (uint32_t g = 0; g < (uint32_t)NG && first + g < count; ++g) {
        const uint32_t pidx = (uint32_t)__builtin_amdgcn_readfirstlane((int)list[first + g]);
        const ewfa_pair_t pg = a.pairs[pidx];
        bp_finish<GL, W>(a, pidx, pg, bp_load(a, pg, GL * W), (int)g * GL, rec, tok, tiles, lane);
    }
}

}  // namespace

// Persistent, one wave per block.  The list holds the pairs class by class,
// widest band first (BP_CLASSES classes from seg[c], seg[BP_CLASSES] the end),
// each by decreasing length; an item is the 64/GL pairs of a wave.
__global__ __launch_bounds__(64, 4) void bp_kernel(BpArgs a) {
    __shared__ uint2 tiles[TRACE_TILES * TILE_STRIDE];
    const int lane = threadIdx.x;
    if (a.seg[BP_CLASSES] == 0) return;
    uint8_t* slot = a.slots + (size_t)blockIdx.x * a.slot_bytes;
    uint32_t* tok = reinterpret_cast<uint32_t*>(slot);
    uint2* rec = reinterpret_cast<uint2*>(slot + a.tok_bytes);
    for (;;) {
        uint32_t item = wave_take(a.queue, 1u, lane);
        int c = 0;
        uint32_t lo = 0, hi = 0, per = 1;
        for (; c < BP_CLASSES; ++c) {
            lo = a.seg[c];
            hi = a.seg[c + 1];
            per = bp_pairs_per_wave(c);
            const uint32_t items = (hi - lo + per - 1u) / per;
            if (item < items) break;
            item -= items;
        }
        if (c == BP_CLASSES) break;
        const uint32_t first = lo + item * per;
        switch (c) {
            case 0: bp_item<64, 4>(a, a.list, first, hi, rec, tok, tiles, lane); break;
            case 1: bp_item<64, 3>(a, a.list, first, hi, rec, tok, tiles, lane); break;
            case 2: bp_item<64, 2>(a, a.list, first, hi, rec, tok, tiles, lane); break;
            case 3: bp_item<64, 1>(a, a.list, first, hi, rec, tok, tiles, lane); break;
            case 4: bp_item<32, 1>(a, a.list, first, hi, rec, tok, tiles, lane); break;
            default: bp_item<16, 1>(a, a.list, first, hi, rec, tok, tiles, lane); break;
        }
        group_sync<1>();
    }
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

// One column: p0, p1 the window's pattern planes, c0, c1 the text base's masks;
// returns bit 0 of the diagonal-delta-0 vector (of the first row).
__device__ __forceinline__ uint32_t band_column(LaneBand& b, uint64_t p0, uint64_t p1, uint64_t c0, uint64_t c1) {
    const uint64_t eq = ~(p0 ^ c0) & ~(p1 ^ c1);
    const uint64_t xh = (((eq & b.vp) + b.vp) ^ b.vp) | eq;
    const uint64_t ph = b.vn | ~(xh | b.vp);
    const uint64_t mh = b.vp & xh;
    const uint64_t d0 = (uint64_t)((uint32_t)xh | (uint32_t)b.vn);
    const uint64_t xv = (eq | b.vn) >> 1;
    b.vp = mh | ~(xv | ph);
    b.vn = ph & xv;
    return (uint32_t)d0;
}

__device__ __forceinline__ uint64_t sign_mask(uint32_t planes, int i) {
    const int m = (int)(planes << (31 - i)) >> 31;
    return (uint64_t)(int64_t)m;
}

__device__ uint32_t lane_bound(const uint64_t* gp, const uint64_t* gt, int plen, int tlen) {
    const int nwp = (plen + 31) >> 5;
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
    const auto window = [&](const uint32_t (&v)[4], int i) -> uint64_t {
        return (uint64_t)__builtin_amdgcn_alignbit(v[1], v[0], (uint32_t)i) |
               ((uint64_t)__builtin_amdgcn_alignbit(v[2], v[1], (uint32_t)i) << 32);
    };
    const int full = tlen >> 5;
    for (int j = 0; j < full; ++j) {
        uint32_t t0, t1;
        load();
        planes_of(gt[j], t0, t1);
        uint32_t z = 0;
#pragma unroll 16
        for (int i = 0; i < 32; ++i) {
            const uint32_t d0 = band_column(b, window(a, i), window(c, i), sign_mask(t0, i), sign_mask(t1, i));
            z = __builtin_amdgcn_alignbit(d0, z, 1);
        }
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
    }
    const int rest = tlen & 31;
    if (rest) {
        uint32_t t0, t1;
        load();
        planes_of(gt[full], t0, t1);
        for (int i = 0; i < rest; ++i)
            b.sc += 1 - (int)(band_column(b, window(a, i), window(c, i), sign_mask(t0, i), sign_mask(t1, i)) & 1u);
        b.r0 += rest;
    }
    // row plen - 1 of the last column
    const int idx = plen - b.r0;
    if (idx <= 0) return (uint32_t)(b.sc - idx);
    const uint64_t m = idx >= 64 ? ~0ull : (1ull << idx) - 1ull;
    return (uint32_t)(b.sc + __popcll(b.vp & m) - __popcll(b.vn & m) + max(idx - 64, 0));
}

}  // namespace

__global__ __launch_bounds__(64, 4) void bp_bound_kernel(const uint64_t* words, const ewfa_pair_t* pairs, uint32_t max_len,
                                                         uint32_t* bound, const uint32_t* list,
                                                         const uint32_t* count_ptr, uint32_t count) {
    const uint32_t n = count_ptr ? *count_ptr : count;
    for (uint32_t item = blockIdx.x * 64u + threadIdx.x; item < n; item += gridDim.x * 64u) {
        const uint32_t pidx = list ? list[item] : item;
        const ewfa_pair_t pr = pairs[pidx];
        uint32_t u = BOUND_NONE;
        if (pr.plen <= max_len && pr.tlen <= max_len)
            u = lane_bound(words + pr.pattern_off, words + pr.text_off, (int)pr.plen, (int)pr.tlen);
        bound[pidx] = u;
    }
}

hipError_t launch_bp_bound(const BpArgs& a, uint32_t* bound, const uint32_t* list, const uint32_t* count_ptr,
                           uint32_t count, uint32_t max_grid, hipStream_t stream) {
    if (count == 0) return hipSuccess;
    const uint32_t blocks = (count + 63u) / 64u;
    hipLaunchKernelGGL(bp_bound_kernel, dim3(blocks < max_grid ? blocks : max_grid), dim3(64), 0, stream, a.words,
                       a.pairs, a.max_len, bound, list, count_ptr, count);
    return hipGetLastError();
}

// ---- which pairs come here -----------------------------------------------------

namespace {

// The class of a pair with distance bound u: the narrowest band that holds
// every path of u edits, or BP_CLASSES for the wavefront (no bound, no band wide
// enough, or so few edits that the wavefront is cheaper).
__device__ __forceinline__ int bp_class_of(const BpArgs& a, const ewfa_pair_t& pr, uint32_t u) {
    if (u == BOUND_NONE || pr.plen > a.max_len || pr.tlen > a.max_len || pr.tlen == 0u || pr.plen == 0u)
        return BP_CLASSES;
    const int tk = (int)pr.tlen - (int)pr.plen;
    for (int c = BP_CLASSES - 1; c >= 0; --c) {
        int S;
        if (bp_band(bp_words(c), tk, S) >= (int)u) {
            // wave instructions of either way (the wavefront's weights fitted
            // to calls: 500,000 pairs of 100..10,000 bp at 1..10% edits took 25.1,
            // 20.6, 20.1 and 20.7 ms with 0.22, 0.5, 1 and 2 per u * u)
            const float wfa = 0.6f * (float)u * (float)u + 100.0f * (float)u;
            const float bp = (float)pr.tlen * (bp_column_cost(c) + 4.0f) + 25.0f * (float)u;
            return wfa < bp ? BP_CLASSES : c;
        }
    }
    // A bound beyond the widest band mostly comes of a window that lost the
    // path at a long gap (values then grow at the rate of unrelated sequences,
    // several times that of 10..15% edits): the distance is likely within the
    // band, and a pair whose is not has wasted little next to the wavefront
    // passes it goes on to.
    int S;
    return bp_band(bp_words(0), tk, S) >= 0 ? 0 : BP_CLASSES;
}

// Bin of a pair in the sort: its class, then its length, longest first.
__device__ __forceinline__ int bp_bin_of(const BpArgs& a, uint32_t pidx, uint32_t u) {
    const ewfa_pair_t pr = a.pairs[pidx];
    const int c = bp_class_of(a, pr, u);
    const uint32_t b = min((uint32_t)((uint64_t)pr.tlen * BP_LEN_BINS / (a.max_len + 1u)), (uint32_t)BP_LEN_BINS - 1u);
    return c * BP_LEN_BINS + (int)(BP_LEN_BINS - 1u - b);
}

}  // namespace

// Counts the list's pairs per bin.
__global__ __launch_bounds__(256) void bp_count_kernel(BpArgs a, const uint32_t* list, const uint32_t* count_ptr,
                                                       uint32_t count) {
    __shared__ uint32_t h[BP_BINS];
    const uint32_t n = count_ptr ? *count_ptr : count;
    const uint32_t base = blockIdx.x * 256u;
    if (base >= n) return;
    for (int i = threadIdx.x; i < BP_BINS; i += 256) h[i] = 0u;
    __syncthreads();
    const uint32_t at = base + threadIdx.x;
    if (at < n) {
        const uint32_t pidx = list ? list[at] : at;
        atomicAdd(&h[bp_bin_of(a, pidx, a.bound[pidx])], 1u);
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
    constexpr int FIRST_REST = BP_CLASSES * BP_LEN_BINS;
    for (int i = threadIdx.x; i < BP_BINS; i += 256) h[i] = 0u;
    if (threadIdx.x == 0) {
        uint32_t run = 0;
        for (int i = 0; i < BP_BINS; ++i) {
            if (i == FIRST_REST) run = 0;
            at[i] = run;
            if (blockIdx.x == 0 && i < FIRST_REST && i % BP_LEN_BINS == 0) a.seg[i / BP_LEN_BINS] = run;
            run += a.bins[i];
            if (blockIdx.x == 0 && i == FIRST_REST - 1) a.seg[BP_CLASSES] = run;
        }
        if (blockIdx.x == 0) *a.rest_count = run;
    }
    __syncthreads();
    const uint32_t item = base + threadIdx.x;
    int b = -1;
    uint32_t pidx = 0, local = 0;
    if (item < n) {
        pidx = list ? list[item] : item;
        b = bp_bin_of(a, pidx, a.bound[pidx]);
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
    hipLaunchKernelGGL(bp_count_kernel, dim3(blocks), dim3(256), 0, stream, a, list, count_ptr, count);
    hipLaunchKernelGGL(bp_place_kernel, dim3(blocks), dim3(256), 0, stream, a, list, count_ptr, count);
    return hipGetLastError();
}

hipError_t launch_bp(const BpArgs& a, uint32_t grid, hipStream_t stream) {
    if (grid == 0) return hipSuccess;
    hipLaunchKernelGGL(bp_kernel, dim3(grid), dim3(64), 0, stream, a);
    return hipGetLastError();
}

int bp_blocks_per_cu() {
    int blocks = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, reinterpret_cast<const void*>(&bp_kernel), 64, 0) !=
        hipSuccess)
        return 0;
    return blocks;
}

}  // namespace ewfa
