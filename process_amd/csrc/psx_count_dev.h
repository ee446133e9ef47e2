// Count-only sequencing on gfx950. Included once, by psx_seq.hip, after
// psx_seq_dev.h.
//
// Two forms with the same counts: k_count_sparse for tables whose records
// reads rarely cover, k_count_dense for the others.
//
// Dense. A block takes a window of one to eight strata of a segment, draws their
// templates in rounds of about 5,600 reads and drops every read, one 32-bit
// word, into the LDS bin of its start (start inside the bin | source copy);
// then the window's records are dealt to the threads, several threads to a
// record, and each scans the bins that can hold reads over its record's
// position: two compares per read, the counts in registers. A read is
// handled once when it is drawn and once per record near it, with no walk, no
// queue and no LDS counters.
//
// Bound by vector instruction issue (4.4 cycles each; 6 waves per SIMD by
// 80 VGPRs and 52 KB of LDS per block; 4 waves: 8.8 ms): on the plain-large
// workload (200x, one record per 200 bases) 325 instructions per 64 templates
// against 497 of a form that walked each read's records and queued (read,
// record) pairs: 80 of them Philox, 80 the rest of the draw and the bins, 35
// the window's set-up, 45 the scan, 80 the errors past their draw. 9.10 ->
// 7.11 ms per 1.6e9 reads, 4.5 ms without errors; 10x single-end reads over
// 300 Mb in windows of 8 strata 1.05 -> 0.57 ms.
//
// A template whose errors its first draw does not settle (more than three of
// them, or two at one base) takes the whole wave 250 instructions; where such
// templates are more than a few in a thousand (the form with MANY) they wait
// in LDS until 48 are there, and each lane makes one's errors.
//
// Sources are cells of the sample, not leaves: the cells that carry a record
// are a range of the sample's cells (cells_below of its leaf range), so a
// template needs no look-up of its leaf. Sequencing errors are drawn per
// template, as in the model; an error matters only where a record lies, which
// a bitmap of the window's record positions tells, and corrects the counts
// there (error_fix).
#pragma once
#include "psx_seq_dev.h"

namespace psxk {

constexpr uint32_t DENSE_BLOCK = 512;
constexpr uint32_t DENSE_WAVES = DENSE_BLOCK / 64;
constexpr uint32_t BIN_SHIFT = 7;     // bins of 128 << lns starts (fewer where the chromosome has fewer than 8,192)
constexpr uint32_t BIN_CAP = 120;     // reads a bin holds; the few beyond it are walked one by one
constexpr uint32_t BIN_STRIDE = BIN_CAP + 4;  // words of a bin: those beyond it land in a slot nobody reads
constexpr uint32_t BIN_READS = 88;    // expected reads of a bin in a round
constexpr uint32_t MAX_BINS = (PSX_STRATUM + MAX_READ) >> BIN_SHIFT;

// Dynamic LDS of a launch: the bitmap of record positions, the bins, their counts (two sets).
constexpr uint32_t MAX_BITS = (PSX_STRATUM << 2) + MAX_READ;  // jobs with errors: windows of at most 4 strata
__host__ __device__ constexpr uint32_t dense_bit_words(uint32_t bits) { return (bits + 127u) / 128u * 4u; }
__host__ __device__ constexpr uint32_t dense_lds(uint32_t bins, uint32_t bits) {
    return 4u * (dense_bit_words(bits) + bins * (BIN_STRIDE + 2u));
}

// The job's insert-size table in LDS: the thresholds and, per guide bucket,
// the first and the last answer a draw of the bucket can have (one word).
constexpr uint32_t COUNT_GUIDE_BITS = 10;
struct count_tables {
    uint32_t ins[MAX_INS];
    uint32_t guide[1u << COUNT_GUIDE_BITS];
};

template <uint32_t BLOCK>
__device__ __forceinline__ void load_count_tables(const job_dev& J, count_tables& t, uint32_t tid) {
    constexpr uint32_t G = 1u << COUNT_GUIDE_BITS, STEP = 1u << (PSX_GUIDE_BITS - COUNT_GUIDE_BITS);
    if (!J.pe) return;
    for (uint32_t i = tid; i < J.ins_n; i += BLOCK) t.ins[i] = J.ins_T[i];
    for (uint32_t i = tid; i < G; i += BLOCK)
        t.guide[i] = (uint32_t)J.ins_guide[i * STEP] |
                     (i + 1u < G ? (uint32_t)J.ins_guide[(i + 1u) * STEP] : J.ins_n - 1u) << 16;
}

// Insert-size pick (psx_guided_pick). Nearly every bucket holds at most one
// threshold, so one compare settles it; where a lane's bucket holds more (the
// tails: one wave in five), a binary search inside the buckets.
__device__ __forceinline__ uint32_t pick_insert(const count_tables& t, uint32_t u) {
    const uint32_t g = t.guide[u >> (32u - COUNT_GUIDE_BITS)];
    uint32_t lo = g & 0xFFFFu, hi = g >> 16;
    const uint32_t first = t.ins[lo];  // lo < hi <= MAX_INS - 1, or the answer
    const bool past = lo < hi && u >= first;
    lo += past ? 1u : 0u;
    if (__ballot(past && lo < hi)) {
        hi = past ? hi : lo;
        while (__ballot(lo < hi)) {
            const uint32_t mid = (lo + hi) >> 1;
            const bool below = u < t.ins[mid], on = lo < hi;
            hi = on && below ? mid : hi;
            lo = on && !below ? mid + 1u : lo;
        }
    }
    return lo;
}

// A descriptor to be read again where it is used: the fields of the rare paths
// are then loaded there instead of being held in scalar registers through the
// hot loop, whose own values they would push into vector lanes.
template <class T>
__device__ __forceinline__ const T& reread(const T& x) {
    uint64_t a = (uint64_t)(uintptr_t)&x;
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+s"(a));
    return *(const T*)(const __attribute__((address_space(4))) T*)a;
#else
    return *(const T*)(uintptr_t)a;
#endif
}

// The records of a window in global memory.
__device__ __forceinline__ glb_view window_view(const job_dev& J, const seg_dev& S, uint32_t k0, uint32_t n) {
    const uint64_t o = out_off(J, S) + k0;
    return glb_view{J.pos + k0, J.lo + k0, J.hi + k0, J.info + k0, J.alt + o, J.depth + o, n};
}

__device__ __forceinline__ uint32_t leaf_of_cell(const job_dev& J, const seg_dev& S, uint32_t cell) {
    return cell == S.n_cells || S.n_cells == 0 ? J.n_leaves : J.sample_leaves[S.leaf_off + cell];
}

// Rare work of a round, listed in LDS and done after its draws: an error of a
// read at a position that holds a record, or a read whose bin is full.
struct todo {
    uint32_t at;    // position of the error or start of the read in the window | substitution << 18 | TODO_READ
    uint32_t copy;  // the source copy
};
constexpr uint32_t TODO_READ = 1u << 20, TODO_POS = (1u << 18) - 1u;
constexpr uint32_t TODO_CAP = 512;  // entries of a round; the ones beyond are done at once

// The rare paths are functions of their own, called: inlined, their loops took
// the scalar registers of the hot loop, which then read its own values back
// from vector lanes (about 55 vector instructions per 64 templates).

__device__ __attribute__((noinline)) void dense_todo(const job_dev* Jp, const seg_dev* Sp, todo T, uint32_t wb,
                                                     uint32_t k0, uint32_t n_win, uint32_t cb) {
    const job_dev& J = *Jp;
    const seg_dev& S = *Sp;
    const glb_view gv = window_view(J, S, k0, n_win);
    const uint32_t P = wb + (T.at & TODO_POS);
    const uint32_t al = T.copy >> cb, leaf = leaf_of_cell(J, S, T.copy & ((1u << cb) - 1u));
    uint32_t i = gv.first(P);
    if (!(T.at & TODO_READ)) {
        error_fix(J, gv, i, al, leaf, (T.at >> 18) & 3u);
    } else {
        while (i < n_win && gv.pos[i] < P + J.L) i = count_group(J, gv, i, al, leaf, terr{0u, 0u}, 0u);
    }
}

// Errors of a slow template into list; returns their number (all lanes of a wave call it).
__device__ __attribute__((noinline)) uint32_t dense_one_slow(const job_dev* Jp, uint32_t r, uint32_t j, uint32_t c2,
                                                         uint32_t* list) {
    const job_dev& J = *Jp;
    wave_sync();
    const uint32_t s0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)J.seed);
    const uint32_t s1 = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(J.seed >> 32));
    const uint32_t n =
        wave_template_errors<true>((uint64_t)s1 << 32 | s0, J.err_n, J.err_k0, J.err_N, J.err_T, r, j, c2, list, threadIdx.x & 63u);
    wave_sync();
    return n;
}

// The errors of a slow template per lane (template r, lanes with on): the
// first K words of its stream that name different bases, in order, f(base
// index, substitution) for each. Returns the lanes with more than MOST (number),
// whose errors the wave has to make (wave_template_errors). A wave's lanes take
// about 44 + 2 MOST vector instructions a word, so some ten for each slow
// template of 48, where the wave's own pass takes 250 for one.
template <uint32_t MOST, class F>
__device__ __forceinline__ unsigned long long lane_errors(const job_dev& J, uint64_t seed, uint32_t r, uint32_t j, uint32_t c2,
                                                          bool on, uint32_t& number, const F& f) {
    psx_u4 w = psx_draw_u(seed, r, j, c2, PSX_P_ERROR << 24);
    uint32_t lo = 0, hi = on ? J.err_n - 1u : 0u;  // thresholds at or below the count's word
    while (__ballot(lo < hi)) {
        if (lo < hi) {
            const uint32_t mid = (lo + hi) >> 1;
            if (w.y >= J.err_T[mid]) lo = mid + 1u; else hi = mid;
        }
    }
    const uint32_t all = on ? J.err_k0 + lo : 0u, K = all > MOST ? 0u : all;
    number = all;
    uint32_t c[MOST], cnt = 0;
#pragma unroll
    for (uint32_t i = 0; i < MOST; ++i) c[i] = 0xFFFFFFFFu;
    for (uint32_t t = 0; t < 4u * PSX_ERR_KCAP && __ballot(cnt < K); ++t) {
        const uint32_t i4 = (t - 3u) & 3u;
        if (t >= 3u && i4 == 0u) w = psx_draw_u(seed, r, j, c2, (PSX_P_ERROR << 24) | (1u + ((t - 3u) >> 2)));
        const uint32_t word = t < 3u ? (t == 0u ? w.x : (t == 1u ? w.z : w.w))
                                     : (i4 == 0u ? w.x : (i4 == 1u ? w.y : (i4 == 2u ? w.z : w.w)));
        const uint32_t x = psx_mulhi32(word, J.err_N);
        bool take = cnt < K;
#pragma unroll
        for (uint32_t i = 0; i < MOST; ++i) take = take & (c[i] != x);
#pragma unroll
        for (uint32_t i = 0; i < MOST; ++i) c[i] = take & (i == cnt) ? x : c[i];
        cnt += take ? 1u : 0u;
        if (take) f(x, ((word & 0xFFFFu) * 3u) >> 16);
    }
    return __ballot(all > MOST);
}

// A wave's slow templates that wait (index, copy, start, mate 2's offset of each), and its stratum and window, kept in LDS
// so that the calls below take no registers of the hot loop.
constexpr uint32_t SLOW_CAP = 48;
static_assert(4 * SLOW_CAP <= ELIST, "the waiting templates take the place of one's errors");
struct slow_list {
    uint32_t list[ELIST];
    uint32_t n, j, c2, wb, k0, n_win, cb, pad;
    const uint32_t* bits;
    uint64_t pad2;
};

struct one_list {
    uint32_t list[ELIST];
};

// The errors of the waiting templates, corrected where they meet a record of the window; all lanes of a wave call it.
__device__ __attribute__((noinline)) void dense_slow(const job_dev* Jp, const seg_dev* Sp, slow_list* l) {
    wave_sync();
    const uint32_t n = l->n, j = l->j, c2 = l->c2, wb = l->wb, k0 = l->k0, n_win = l->n_win, cb = l->cb;
    const uint32_t* const bits = l->bits;
    uint32_t* const list = l->list;
    const job_dev& J = *Jp;
    const uint32_t lane = threadIdx.x & 63u;
    const bool on = lane < n;
    const uint4 T = ((const uint4*)list)[on ? lane : 0u];  // index, copy, start, offset
    wave_sync();  // every entry read: the list is free
    if (lane == 0) l->n = 0;
    const uint32_t s0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)J.seed);
    const uint32_t s1 = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(J.seed >> 32));
    const uint64_t seed = (uint64_t)s1 << 32 | s0;
    const uint32_t RL = J.L;
    auto error = [&](uint32_t x, uint32_t d, uint32_t X, uint32_t bi, uint32_t sub) {
        const uint32_t p = bi + (bi >= RL ? x + d - RL : x);
        if ((bits[p >> 5] >> (p & 31u)) & 1u) dense_todo(Jp, Sp, todo{p | sub << 18, X}, wb, k0, n_win, cb);
    };
    uint32_t number;
    unsigned long long big =
        lane_errors<8>(J, seed, T.x, j, c2, on, number, [&](uint32_t bi, uint32_t sub) { error(T.z, T.w, T.y, bi, sub); });
    while (big) {
        const int ln = __ffsll((long long)big) - 1;
        big &= big - 1ull;
        const uint32_t rs = (uint32_t)__builtin_amdgcn_readlane((int)T.x, ln), Xs = (uint32_t)__builtin_amdgcn_readlane((int)T.y, ln);
        const uint32_t xs = (uint32_t)__builtin_amdgcn_readlane((int)T.z, ln), ds = (uint32_t)__builtin_amdgcn_readlane((int)T.w, ln);
        const uint32_t ne = wave_template_errors<true>(seed, J.err_n, J.err_k0, J.err_N, J.err_T, rs, j, c2, list, lane,
                                                 (uint32_t)__builtin_amdgcn_readlane((int)number, ln));
        wave_sync();
        for (uint32_t k = lane; k < ne; k += 64u) error(xs, ds, Xs, list[k] & 0xFFFFFu, list[k] >> 20);
        wave_sync();
    }
}

// The slow templates of a group (lanes of the mask) wait until SLOW_CAP are there.
__device__ __attribute__((noinline)) void dense_wait(const job_dev* Jp, const seg_dev* Sp, slow_list* l, unsigned long long slow,
                                                     uint32_t r, uint32_t X, uint32_t x, uint32_t d) {
    const uint32_t lane = threadIdx.x & 63u;
    while (slow) {
        const uint32_t n = (uint32_t)__builtin_amdgcn_readfirstlane((int)l->n);
        const uint32_t at =
            n + __builtin_amdgcn_mbcnt_hi((uint32_t)(slow >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)slow, 0u));
        const bool in = ((slow >> lane) & 1ull) && at < SLOW_CAP;
        if (in) ((uint4*)l->list)[at] = uint4{r, X, x, d};
        const unsigned long long m = __ballot(in);
        slow &= ~m;
        if (lane == 0) l->n = n + (uint32_t)__popcll(m);
        wave_sync();
        if (n + (uint32_t)__popcll(m) == SLOW_CAP) dense_slow(Jp, Sp, l);
        wave_sync();
    }
}

// The reads of one bin over a record that shares its position (or has no single range of carriers).
__device__ __attribute__((noinline)) void dense_group(const job_dev* Jp, const seg_dev* Sp, const uint32_t* bin,
                                                      uint32_t k, uint32_t n, uint32_t step, uint32_t elo, uint32_t elen,
                                                      uint32_t lw, uint32_t cb, uint32_t k0, uint32_t n_win, uint32_t i) {
    const job_dev& J = *Jp;
    const seg_dev& S = *Sp;
    const glb_view gv = window_view(J, S, k0, n_win);
    for (; k < n; k += step) {
        const uint32_t w = bin[k];
        if (w - elo > elen) continue;
        const uint32_t X = w & (0xFFFFFFFFu >> lw);
        count_group(J, gv, i, X >> cb, leaf_of_cell(J, S, X & ((1u << cb) - 1u)), terr{0u, 0u}, 0u);
    }
}

// The templates [t0, t1) of the item's part of stratum [b, e) (wave-uniform; all lanes of the wave call it).
__device__ __forceinline__ void wave_share(const seg_dev& S, uint32_t part, uint32_t b, uint32_t e, uint32_t lane,
                                           uint32_t& t0, uint32_t& t1) {
    const uint32_t below = (uint32_t)templates_below(S, lane ? e : b);  // lane 0: its first template; lane 1: its end
    const uint32_t nj = (uint32_t)__builtin_amdgcn_readlane((int)below, 1) -
                        (uint32_t)__builtin_amdgcn_readfirstlane((int)below);
    t0 = 0;
    t1 = nj;
    if (seg_parts(S) != 1u) {
        const uint32_t share = (nj + seg_parts(S) - 1u) / seg_parts(S);
        t0 = min(nj, part * share);
        t1 = min(nj, t0 + share);
    }
}

// The descriptor a wave-uniform pointer argument names, read with scalar loads.
template <class T>
__device__ __forceinline__ const T& uniform_ref(const T* p) {
    const uint64_t a = (uint64_t)(uintptr_t)p;
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(a >> 32));
#if defined(__HIP_DEVICE_COMPILE__)
    return *(const T*)(const __attribute__((address_space(4))) T*)((uint64_t)hi << 32 | lo);
#else
    return *(const T*)(uintptr_t)((uint64_t)hi << 32 | lo);
#endif
}

// A template of any ploidy and any copy-number events; out of line, so that its registers are not the loops'.
struct general_draw {
    uint32_t x, cell, allele, ins;
    uint32_t kept;  // a word of its own: the allele of a draw that is not kept is any copy slot
};
template <bool CNA>
__device__ __attribute__((noinline)) general_draw draw_general(const job_dev* J, const seg_dev* S, uint32_t r, uint32_t j,
                                                               uint32_t b, uint32_t e) {
    psx_u4 w;
    const tmpl t = template_source<CNA, false>(uniform_ref(J), uniform_ref(S), r, j, b, e, w);
    return general_draw{t.x, t.cell, t.allele, w.w, t.ok};
}

// What a segment's template draws use, read once per item. A diploid source
// without copy-number events is drawn here, any other by template_source.
struct source_draw {
    uint32_t n_cells, copies, normal_below, starts_end, RL;
    int ins_past;  // the smallest insert size over the read size
    bool diploid, normal_some;
    __device__ __forceinline__ source_draw(const job_dev& J, const seg_dev& S, bool cna)
        : n_cells(S.n_cells), copies(S.n_cells ? 2u * S.n_cells : 2u), normal_below((uint32_t)(J.thr_normal - 1u)),
          starts_end(S.len - J.L), RL(J.L), ins_past((int)J.ins_k0 - (int)J.L),
          diploid(J.ploidy == 2u && !(cna && S.n_cna != 0u)), normal_some(S.n_cells != 0u && J.thr_normal != 0u) {}
    // Template r of stratum j = [b, e): start in the window that begins at wb, source cell (n_cells: the normal genome)
    // and allele, and the word that gives its insert size; false when a copy-number draw rejects it. cw: the window's
    // n_ev copy-number events (CN_GENERAL: none listed).
    template <bool CNA>
    __device__ __forceinline__ bool draw(const job_dev& J, const seg_dev& S, const cn_window* cw, uint32_t n_ev, uint32_t r,
                                         uint32_t j, uint32_t c2, uint32_t b, uint32_t e, uint32_t wb, uint32_t& x,
                                         uint32_t& ins, uint32_t& cell, uint32_t& al) const {
        psx_u4 w;
        bool ok = true;
        if (CNA && n_ev != CN_GENERAL) {
            w = psx_draw_u(J.seed, r, j, c2, PSX_P_TEMPLATE << 24);
            x = b + psx_uniform32(w.x, e - b);
            ok = cn_source(S, *cw, n_ev, normal_some && w.y <= normal_below, w.z, x, cell, al);
            x -= wb;
        } else if (diploid) {
            w = psx_draw_u(J.seed, r, j, c2, PSX_P_TEMPLATE << 24);
            x = b - wb + psx_uniform32(w.x, e - b);
            uint32_t v = psx_uniform32(w.z, copies);
            cell = v >> 1;
            if (normal_some) {
                const bool normal = w.y <= normal_below;
                v = normal ? w.z >> 31 : v;
                cell = normal ? n_cells : cell;
            }
            al = v & 1u;
        } else {
            const general_draw t = draw_general<CNA>(&J, &S, r, j, b, e);
            x = t.x - wb;
            cell = t.cell;
            al = t.allele;
            ok = t.kept != 0u;
            w.w = t.ins;
        }
        ins = w.w;
        return ok;
    }
    // Mate 2's offset from the start.
    __device__ __forceinline__ uint32_t offset(const job_dev& J, const count_tables& tab, uint32_t ins, uint32_t wb,
                                               uint32_t x) const {
        if (!J.pe) return 0;
        const int I = (int)pick_insert(tab, ins) + ins_past;
        return min((uint32_t)max(I, 0), starts_end - wb - x);
    }
};

// Copy-number draws reject templates: the accepted ones are packed into the lanes of a pending set, which takes the
// place of a group when the next would overflow it (and at the end).
struct pending {
    uint32_t n = 0, x = 0, ins = 0, copy = 0, r = 0;
    // The group's values (of the lanes that are on) go in; true: the set's come out, of its first lanes, and x is 0 in
    // the others.
    __device__ __forceinline__ bool pack(bool more, bool& on, uint32_t lane, uint32_t& gx, uint32_t& gi, uint32_t& gc,
                                         uint32_t& gr) {
        const unsigned long long m = __ballot(on);
        const uint32_t k = (uint32_t)__popcll(m), had = n;
        const bool out = n + k > 64u || !more;
        const uint32_t at = out ? 0u : n;
        const uint32_t below = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
        const int to = (int)((on ? at + below : (at + k + (lane - below)) & 63u) * 4u);
        const uint32_t nx = (uint32_t)__builtin_amdgcn_ds_permute(to, (int)gx);
        const uint32_t ni = (uint32_t)__builtin_amdgcn_ds_permute(to, (int)gi);
        const uint32_t nc = (uint32_t)__builtin_amdgcn_ds_permute(to, (int)gc);
        const uint32_t nr = (uint32_t)__builtin_amdgcn_ds_permute(to, (int)gr);
        on = out && lane < had;
        gx = on ? x : 0u;
        gi = ins;
        gc = copy;
        gr = on ? r : (uint32_t)__builtin_amdgcn_readfirstlane((int)r);
        const bool recv = lane - at < k;
        x = recv ? nx : x;
        ins = recv ? ni : ins;
        copy = recv ? nc : copy;
        r = recv ? nr : r;
        n = at + k;
        return out && had != 0u;
    }
};

// The carriers of record q among the reads of the segment's sample: cells [lo, lo + len) (the normal genome is cell
// n_cells); false when they are no single range.
__device__ __forceinline__ bool carrier_cells(const job_dev& J, const seg_dev& S, uint64_t q, uint32_t info, uint32_t& lo,
                                              uint32_t& len) {
    const uint32_t nat = PSX_INFO_NATURE(info);
    const bool normal_has = nat == PSX_GERMINAL || (nat == PSX_PRENEOPLASTIC && J.preneo);
    lo = 0;
    uint32_t hi = normal_has ? 1u : 0u;  // the normal sample: one cell
    bool one_range = true;
    if (S.n_cells) {
        lo = cells_below(J, S.sample, J.lo[q]);
        hi = cells_below(J, S.sample, J.hi[q]);
        if (normal_has && J.thr_normal) {  // reads of the normal genome carry it too
            one_range = hi == S.n_cells || lo == hi;
            lo = lo == hi ? S.n_cells : lo;
            hi = S.n_cells + 1u;
        }
    }
    len = hi - lo;
    return one_range;
}

// Whether the carrier range decides an alternative read of a record alone at its position.
__device__ __forceinline__ bool plain_record(uint32_t info) {
    return PSX_INFO_HEAD(info) && (PSX_INFO_KIND(info) != PSX_SNV || PSX_INFO_REF(info) != PSX_INFO_ALT(info));
}

// ------------------------------------------------- tables with few mutations
//
// Where reads rarely cover a record, a template ends with one test per read:
// a bit per 8 starts of the window says whether a read that starts there can
// reach a record. The reads that can are queued by the wave and counted 64 at
// a time, one per lane: the records each covers, found in LDS, the carriers as
// ranges of the sample's cells, and the errors of its template, drawn only
// then. Bound by vector instruction issue: 115 instructions per 64 templates
// where nothing is covered (43 Philox, 20 the source, 20 the insert size, 20
// the tests; 4.4-4.7 cycles each), and about 390 per 64 queued reads. The form
// before walked every read's records and queued positions: 200 Mb at 30x with
// one record per 13,000 bases 559 -> 357 us, 1.5 Mb at 2000x 500 -> 447 us.
// With a bit per 32 starts instead of 8 (more reads queued in vain) 362 and
// 486 us.
//
// A queued read whose template's errors its first draw does not settle is
// counted without them, and the wave makes them, 250 vector instructions a
// template; where such templates are many (the form with MANY) the reads wait
// until 48 do, and each lane makes one's: 2.8e7 reads of 250 bases at 0.8 %
// 1.38 -> 0.50 ms, pairs of 150 at 2 % 6.6 -> 1.4 ms.

// An entry of a wave's queue: a read.
struct sparse_read {
    uint32_t at;    // start in the window | mate << 18 | allele << 19
    uint32_t cell;  // its source cell (the normal genome: n_cells)
    uint32_t r;     // template index
};

constexpr uint32_t START_SHIFT = 3;  // starts per bit of the reach bitmap
constexpr uint32_t WAIT_FULL = 48;  // reads that wait before their templates' errors are made, and room for a queue's more
constexpr uint32_t WAIT_READS = WAIT_FULL + 64;

template <int BLOCK, int CAP, bool MANY>
struct sparse_lds {
    static constexpr uint32_t WAVES = BLOCK / 64;
    static constexpr bool SLOW_WAIT = MANY;
    static constexpr uint32_t START_BITS = ((PSX_STRATUM * WAVES + MAX_READ) >> START_SHIFT) + 1u;
    count_tables tab;
    uint32_t err[4];                         // thresholds of 1 to 4 errors, padded
    uint32_t p[CAP], low[CAP], len[CAP], info[CAP];  // records: position in the window, cells [low, low + len)
    uint32_t dep[CAP], alt[CAP];
    uint32_t bits[(START_BITS + 31u) / 32u];
    sparse_read queue[WAVES][128];
    sparse_read wait[WAVES][MANY ? WAIT_READS : 1u];  // counted reads of slow templates, whose errors are not made yet
    uint32_t wait_n[WAVES];
    uint32_t run, acc;
};
static_assert(64 * sizeof(sparse_read) >= 4 * ELIST, "a slow template's errors take the place of the entries counted");

// info word of a staged record: the table's, with bits 30 (counted with the first record of its position) and 31 (that
// first record, or one whose carriers are no single range) set where the record is not counted alone
constexpr uint32_t REC_SKIP = 1u << 30, REC_SHARED = 1u << 31;

// The queued reads q[0, n) of a wave, one per lane; n_lds: records staged (0: the window has more, all in global memory).
template <class LDS>
__device__ __forceinline__ void stage_record(const job_dev& J, const seg_dev& S, LDS& lds, uint32_t k0, uint32_t i,
                                             uint32_t p) {
    const uint32_t q = k0 + i;
    const uint32_t info = J.info[q];
    uint32_t lo, len;
    const bool one_range = carrier_cells(J, S, q, info, lo, len);
    uint32_t flag = 0;
    if (!PSX_INFO_SOLO(info)) flag = i > 0 && J.pos[q - 1] == J.pos[q] ? REC_SKIP : REC_SHARED;
    else if (!one_range || !plain_record(info)) flag = REC_SHARED;
    lds.p[i] = p;
    lds.low[i] = lo;
    lds.len[i] = len;
    lds.info[i] = (info & ~(REC_SKIP | REC_SHARED)) | flag;
}

// The errors of the slow templates of the last 64 reads that wait: each lane makes one's, up to 16 of them (lane_errors), and corrects
// the counts at those on the read that meet a record; the wave makes the others', one template after another (in list,
// ELIST words), or two at a time where they have up to PAIR_ERRORS (7e6 reads of 1,000 bases at 2 %: 3.28 -> 2.01 ms). All lanes of a
// wave call it.
constexpr uint32_t PAIR_ERRORS = 28;
template <class LDS>
__device__ __attribute__((noinline)) void count_slow(const job_dev* Jp, const seg_dev* Sp, LDS* lds, uint32_t* list,
                                                     uint32_t wb, uint32_t k0, uint32_t n_win, uint32_t n_lds, uint32_t j,
                                                     uint32_t c2) {
    const job_dev& J = *Jp;
    const seg_dev& S = *Sp;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    wave_sync();
    const uint32_t n = lds->wait_n[wave], from = n > 64u ? n - 64u : 0u;
    const bool on = from + lane < n;
    const sparse_read R = on ? lds->wait[wave][from + lane] : sparse_read{0u, 0u, 0u};
    wave_sync();  // every lane has read its entry
    if (lane == 0) lds->wait_n[wave] = from;
    const uint32_t RL = J.L;
    const uint32_t s0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)J.seed);
    const uint32_t s1 = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(J.seed >> 32));
    const uint64_t seed = (uint64_t)s1 << 32 | s0;
    const glb_view gv = window_view(J, S, k0, n_win);
    uint32_t a0 = 0;  // the read's first record
    for (uint32_t z = on ? n_lds : 0u; a0 < z;) {
        const uint32_t mid = (a0 + z) >> 1;
        if (lds->p[mid] < (R.at & 0x3FFFFu)) a0 = mid + 1u; else z = mid;
    }
    // base index bi of the template of the read (at, cell), whose first record is `first`, substituted
    auto error = [&](uint32_t at, uint32_t cell, uint32_t first, uint32_t bi, uint32_t sub) {
        const uint32_t mate = (at >> 18) & 1u, al = at >> 19;
        if ((bi >= RL ? 1u : 0u) != mate) return;
        const uint32_t p = (at & 0x3FFFFu) + bi - mate * RL;
        if (n_lds) {
            uint32_t a = first;
            while (a < n_lds && lds->p[a] < p) ++a;
            if (a == n_lds || lds->p[a] != p) return;
            const uint32_t in = lds->info[a];
            if (in & REC_SHARED) {
                error_fix(J, gv, a, al, leaf_of_cell(J, S, cell), sub);
            } else if (PSX_INFO_KIND(in) == PSX_SNV) {
                const bool car = PSX_INFO_ALLELE(in) == al && cell - lds->low[a] < lds->len[a];
                const uint32_t alt = PSX_INFO_ALT(in), tb = car ? alt : PSX_INFO_REF(in), ob = sub < tb ? sub : sub + 1u;
                if ((ob == alt) != (tb == alt)) atomicAdd(&lds->alt[a], ob == alt ? 1u : 0xFFFFFFFFu);
            }
        } else {
            const uint32_t a = gv.first(wb + p);
            if (a < n_win && gv.pos[a] == wb + p) error_fix(J, gv, a, al, leaf_of_cell(J, S, cell), sub);
        }
    };
    uint32_t number;
    unsigned long long big = lane_errors<16>(J, seed, R.r, j, c2, on, number,
                                             [&](uint32_t bi, uint32_t sub) { error(R.at, R.cell, a0, bi, sub); });
    // two templates of up to PAIR_ERRORS at a time: the first 32 words of one's stream in each half of the wave
    unsigned long long pairs = __ballot(number > 16u && number <= PAIR_ERRORS);
    big &= ~pairs;
    const uint32_t upper = lane >> 5, t = lane & 31u;
    while (pairs) {
        const int la = __ffsll((long long)pairs) - 1;
        pairs &= pairs - 1ull;
        const bool two = pairs != 0ull;
        const int lb = two ? __ffsll((long long)pairs) - 1 : la;
        pairs &= two ? pairs - 1ull : 0ull;
        const int src = upper ? lb : la;
        const uint32_t at = (uint32_t)__shfl((int)R.at, src), cell = (uint32_t)__shfl((int)R.cell, src);
        const uint32_t rs = (uint32_t)__shfl((int)R.r, src), first = (uint32_t)__shfl((int)a0, src);
        const uint32_t K = (uint32_t)__shfl((int)number, src);
        wave_sync();
        list[lane] = 0;  // 1,024 bits of hashed indices for each half
        wave_sync();
        const psx_u4 w = psx_draw_u(seed, rs, j, c2, (PSX_P_ERROR << 24) | (t < 3u ? 0u : 1u + ((t - 3u) >> 2)));
        const uint32_t word = psx_word(w, t < 3u ? (t == 0u ? 0 : (int)t + 1) : (int)((t - 3u) & 3u));
        const uint32_t x = psx_mulhi32(word, J.err_N), h = (x * 0x9E3779B1u) >> 22, bit = 1u << (h & 31u);
        const bool seen = atomicOr(&list[upper * 32u + (h >> 5)], bit) & bit;
        const unsigned long long half = upper ? 0xFFFFFFFF00000000ull : 0xFFFFFFFFull;
        unsigned long long again = 0;
        for (unsigned long long left = __ballot(seen); left;) {  // of the lanes that name one index all but one found it
            const int ln = __ffsll((long long)left) - 1;
            const uint32_t xq = (uint32_t)__builtin_amdgcn_readlane((int)x, ln);
            const unsigned long long same = __ballot(x == xq && upper == (uint32_t)ln >> 5);
            left &= ~same;
            again |= same & (same - 1ull);
        }
        const unsigned long long fresh = ~again & half;
        const uint32_t n_fresh = (uint32_t)__popcll(fresh), rank = (uint32_t)__popcll(fresh & ((1ull << lane) - 1ull));
        if (n_fresh >= K && (two || !upper) && ((fresh >> lane) & 1ull) && rank < K)
            error(at, cell, first, x, ((word & 0xFFFFu) * 3u) >> 16);
        const unsigned long long few = __ballot(n_fresh < K);  // too many repeats among the 32 words
        big |= few & 1ull ? 1ull << la : 0ull;
        big |= few >> 32 & 1ull ? 1ull << lb : 0ull;
    }
    while (big) {
        const int ln = __ffsll((long long)big) - 1;
        big &= big - 1ull;
        const uint32_t at = (uint32_t)__builtin_amdgcn_readlane((int)R.at, ln), cell = (uint32_t)__builtin_amdgcn_readlane((int)R.cell, ln);
        const uint32_t rs = (uint32_t)__builtin_amdgcn_readlane((int)R.r, ln), first = (uint32_t)__builtin_amdgcn_readlane((int)a0, ln);
        wave_sync();
        const uint32_t ne = wave_template_errors<true>(seed, J.err_n, J.err_k0, J.err_N, J.err_T, rs, j, c2, list, lane,
                                                 (uint32_t)__builtin_amdgcn_readlane((int)number, ln));
        wave_sync();
        for (uint32_t k = lane; k < ne; k += 64u) error(at, cell, first, list[k] & 0xFFFFFu, list[k] >> 20);
    }
    wave_sync();
}

template <class LDS>
__device__ __attribute__((noinline)) void count_queued(const job_dev* Jp, const seg_dev* Sp, LDS* lds,
                                                       sparse_read* q, uint32_t n, uint32_t wb, uint32_t k0,
                                                       uint32_t n_win, uint32_t n_lds, uint32_t j, uint32_t c2) {
    const job_dev& J = *Jp;
    const seg_dev& S = *Sp;
    const uint32_t lane = threadIdx.x & 63u;
    const bool on = lane < n;
    const sparse_read R = on ? q[lane] : sparse_read{0u, 0u, 0u};
    const uint32_t xr = R.at & 0x3FFFFu, mate = (R.at >> 18) & 1u, al = R.at >> 19;
    const uint32_t leaf = on ? leaf_of_cell(J, S, R.cell) : 0u;
    const uint32_t end = xr + J.L, boff = mate * J.L - xr;  // base index of position p in the template: p + boff
    const uint32_t s0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)J.seed);
    const uint32_t s1 = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(J.seed >> 32));
    const glb_view gv = window_view(J, S, k0, n_win);
    terr e{0u, 0u};
    if (J.err_n) e = template_errors(J, (uint64_t)s1 << 32 | s0, lds->err, R.r, j, c2, on);
    if (n_lds) {
        uint32_t a = 0, z = on ? n_lds : 0u;
        while (a < z) {
            const uint32_t mid = (a + z) >> 1;
            if (lds->p[mid] < xr) a = mid + 1; else z = mid;
        }
        for (; on && a < n_lds; ++a) {
            const uint32_t p = lds->p[a];
            if (p >= end) break;
            const uint32_t in = lds->info[a];
            if (in & (REC_SKIP | REC_SHARED)) {
                if (in & REC_SHARED) count_group(J, gv, a, al, leaf, e, boff - wb);
                continue;
            }
            atomicAdd(&lds->dep[a], 1u);
            const bool car = PSX_INFO_ALLELE(in) == al && R.cell - lds->low[a] < lds->len[a];
            bool hit = car;
            if (PSX_INFO_KIND(in) == PSX_SNV) {
                const uint32_t tb = car ? PSX_INFO_ALT(in) : PSX_INFO_REF(in);
                hit = observe(e, p + boff, tb) == PSX_INFO_ALT(in);
            }
            if (hit) atomicAdd(&lds->alt[a], 1u);
        }
    } else if (on) {
        uint32_t i = gv.first(wb + xr);
        while (i < n_win && gv.pos[i] < wb + end) i = count_group(J, gv, i, al, leaf, e, boff - wb);
    }
    // slow templates counted without errors
    unsigned long long sm = __ballot(on && e.slow());
    if constexpr (LDS::SLOW_WAIT) {  // wait (count_slow); there is room for 64
        if (sm) {
            const uint32_t wave = threadIdx.x >> 6, had = lds->wait_n[wave];
            const uint32_t at =
                had + __builtin_amdgcn_mbcnt_hi((uint32_t)(sm >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)sm, 0u));
            if ((sm >> lane) & 1ull) lds->wait[wave][at] = R;
            wave_sync();
            if (lane == 0) lds->wait_n[wave] = had + (uint32_t)__popcll(sm);
        }
        wave_sync();
        return;
    }
    // the wave generates each one's and corrects the counts at those of this mate
    uint32_t* list = (uint32_t*)q;  // every lane has read its entry
    while (sm) {
        const int ln = __ffsll((long long)sm) - 1;
        sm &= sm - 1ull;
        const uint32_t xs = (uint32_t)__builtin_amdgcn_readlane((int)xr, ln), ms = (uint32_t)__builtin_amdgcn_readlane((int)mate, ln);
        const uint32_t as = (uint32_t)__builtin_amdgcn_readlane((int)al, ln), ls = (uint32_t)__builtin_amdgcn_readlane((int)leaf, ln);
        const uint32_t rs = (uint32_t)__builtin_amdgcn_readlane((int)R.r, ln);
        wave_sync();
        const uint32_t ne = wave_template_errors<true>((uint64_t)s1 << 32 | s0, J.err_n, J.err_k0, J.err_N, J.err_T, rs, j, c2, list, lane);
        wave_sync();
        for (uint32_t k = lane; k < ne; k += 64u) {
            const uint32_t w = list[k], bi = w & 0xFFFFFu;
            if ((bi >= J.L ? 1u : 0u) != ms) continue;
            const uint32_t P = wb + xs + bi - ms * J.L;
            const uint32_t i = gv.first(P);
            if (i < n_win && gv.pos[i] == P) error_fix(J, gv, i, as, ls, w >> 20);
        }
    }
    wave_sync();
}

template <int BLOCK, int CAP, bool CNA, bool MANY>
__global__ void __launch_bounds__(BLOCK, 6) k_count_sparse(const seq_launch L) {
    using LDS = sparse_lds<BLOCK, CAP, MANY>;
    __shared__ LDS lds;
    __shared__ cn_window s_cn;  // copy numbers
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    sparse_read* const queue = lds.queue[wave];
    uint32_t in_tab = UNRESOLVED;
    for (uint32_t i = tid; i < (uint32_t)CAP; i += BLOCK) lds.dep[i] = lds.alt[i] = 0;
    for (uint32_t i = tid; i < (LDS::START_BITS + 31u) / 32u; i += BLOCK) lds.bits[i] = 0;
    if (MANY && lane == 0) lds.wait_n[wave] = 0;
    __syncthreads();
    for (uint32_t run = blockIdx.x;;) {
        const item_run R0 = run_of(L, run);
        if (R0.first == R0.end) break;
        if (tid == 0) lds.run = gridDim.x + (uint32_t)atomicAdd(L.queue, 1ull);  // the block's next run
        for (uint32_t item = R0.first; item < R0.end; ++item) {
            const item_dev it = uniform_at(L.items, item);
            const seg_dev& S = *(const seg_dev*)((const __attribute__((address_space(4))) seg_dev*)L.segs + it.seg);
            const job_dev& J = *(const job_dev*)((const __attribute__((address_space(4))) job_dev*)L.jobs + S.job);
            const uint32_t c2 = (S.chr << 16) | S.so;
            const uint32_t lns = seg_lns(S), nslot = LDS::WAVES >> lns, slot = wave & (nslot - 1u);
            const uint32_t RL = J.L, pe = J.pe;
            const source_draw D(J, S, CNA);
            if (CNA && tid == 0) lds.acc = 0;
            if (in_tab != S.job) {
                in_tab = S.job;
                load_count_tables<BLOCK>(J, lds.tab, tid);
                if (tid < 4u) lds.err[tid] = tid < J.err_n ? J.err_T[tid] : 0xFFFFFFFFu;
            }
            uint32_t acc = 0;  // accepted templates (wave-uniform)
            for (uint32_t jw = it.j0; jw < it.j1; jw += 1u << lns) {
                const uint32_t wb = jw * PSX_STRATUM, je = min(jw + (1u << lns), it.j1);
                const uint32_t starts = min(je * PSX_STRATUM, S.W);
                const uint32_t wend = min(S.len, starts - 1u + J.reach);
                const uint32_t k0 = uniform_at(J.bucket, S.bucket_off + jw);
                const uint32_t n_win = window_records(J, S, k0, wend);
                const uint32_t n_lds = n_win <= (uint32_t)CAP ? n_win : 0u;
                if (CNA && S.n_cna && wave == 0) cn_fill(J, S, wb, starts, lane, s_cn);
                // the records, and the starts from which a read reaches one
                for (uint32_t i = tid; i < n_win; i += BLOCK) {
                    const uint32_t p = J.pos[k0 + i] - wb;
                    if (n_lds) stage_record(J, S, lds, k0, i, p);
                    if (p >= wend - wb) continue;
                    const uint32_t f = (p + 1u > RL ? p + 1u - RL : 0u) >> START_SHIFT, l = p >> START_SHIFT;
                    for (uint32_t w = f >> 5; w <= l >> 5; ++w) {
                        const uint32_t from = w == f >> 5 ? f & 31u : 0u, to = w == l >> 5 ? l & 31u : 31u;
                        atomicOr(&lds.bits[w], (0xFFFFFFFFu << from) & (0xFFFFFFFFu >> (31u - to)));
                    }
                }
                __syncthreads();
                const uint32_t j = jw + wave / nslot;
                const uint32_t b = j * PSX_STRATUM, e = min(b + PSX_STRATUM, S.W);
                uint32_t t0 = 0, t1 = 0;
                if (j < je) wave_share(S, it.part, b, e, lane, t0, t1);
                uint32_t qn = 0;
                const uint32_t n_ev = CNA && S.n_cna ? (uint32_t)__builtin_amdgcn_readfirstlane((int)s_cn.n) : CN_GENERAL;
                for (uint32_t g = t0 + slot * 64u; g < t1; g += nslot * 64u) {  // wave-uniform
                    bool on = g + lane < t1;
                    const uint32_t r = on ? g + lane : g;
                    uint32_t x, ins, cell, al;
                    on = D.draw<CNA>(J, S, &s_cn, n_ev, r, j, c2, b, e, wb, x, ins, cell, al) && on;
                    const uint32_t d = D.offset(J, lds.tab, ins, wb, x);
                    if (CNA) acc += (uint32_t)__popcll(__ballot(on));
                    for (uint32_t m = 0; m <= pe; ++m) {
                        const uint32_t xm = m ? x + d : x;
                        const uint32_t bit = xm >> START_SHIFT;
                        const bool add = on && ((lds.bits[bit >> 5] >> (bit & 31u)) & 1u);
                        const unsigned long long mask = __ballot(add);
                        if (!mask) continue;
                        if (add)
                            queue[qn + __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                                                 __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u))] =
                                sparse_read{xm | m << 18 | al << 19, cell, r};
                        qn += (uint32_t)__popcll(mask);
                        if (qn >= 64u) {
                            qn -= 64u;
                            wave_sync();
                            count_queued(&J, &S, &lds, queue + qn, 64u, wb, k0, n_win, n_lds, j, c2);
                            if (MANY && __builtin_amdgcn_readfirstlane((int)lds.wait_n[wave]) >= WAIT_FULL)
                                count_slow(&J, &S, &lds, (uint32_t*)(queue + qn), wb, k0, n_win, n_lds, j, c2);
                        }
                    }
                }
                if (qn) {
                    wave_sync();
                    count_queued(&J, &S, &lds, queue, qn, wb, k0, n_win, n_lds, j, c2);
                }
                while (MANY && __builtin_amdgcn_readfirstlane((int)lds.wait_n[wave]))
                    count_slow(&J, &S, &lds, (uint32_t*)queue, wb, k0, n_win, n_lds, j, c2);
                __syncthreads();
                for (uint32_t i = tid; i < n_lds; i += BLOCK) {
                    const uint32_t dep = lds.dep[i], alt = lds.alt[i];
                    if (dep) {
                        const uint64_t o = out_off(J, S) + k0 + i;
                        atomicAdd(J.depth + o, (int32_t)dep);
                        if (alt) atomicAdd(J.alt + o, (int32_t)alt);
                        lds.dep[i] = lds.alt[i] = 0;
                    }
                }
                for (uint32_t i = tid; i < (((wend - wb) >> START_SHIFT) + 32u) >> 5; i += BLOCK) lds.bits[i] = 0;
                __syncthreads();
            }
            if (CNA && S.n_cna) {
                if (acc && lane == 0) atomicAdd(&lds.acc, acc);
                __syncthreads();
                if (tid == 0 && lds.acc) atomicAdd(J.acc, (unsigned long long)lds.acc * (J.pe + 1u));
            }
        }
        __syncthreads();
        run = __builtin_amdgcn_readfirstlane(lds.run);
        __syncthreads();  // read by every wave before it is written again
    }
}

// ---------------------------------------------- tables with many mutations

// A record as the scan sees it: position in the window, and the carrying
// copies [low, low + len) of the word's copy field (allele above the cell).
// Records alone at their position are counted by the scan alone; one that
// shares its position is counted with it by the first of them (GROUP), as is
// one whose carriers are no single range.
struct scan_rec {
    uint32_t p, low, len, kind;
};
enum : uint32_t { REC_NONE = 0, REC_SOLO = 1, REC_GROUP = 2 };

__device__ __forceinline__ scan_rec load_rec(const job_dev& J, const seg_dev& S, uint32_t wb, uint32_t k0, uint32_t i,
                                             uint32_t cb, uint32_t lw) {
    const uint32_t q = k0 + i;
    const uint32_t pos = J.pos[q], info = J.info[q];
    uint32_t lo, len;
    const bool one_range = carrier_cells(J, S, q, info, lo, len);
    scan_rec R;
    R.p = pos - wb;
    R.low = ((PSX_INFO_ALLELE(info) << cb) | lo) << lw;
    R.len = len << lw;
    if (PSX_INFO_SOLO(info)) R.kind = one_range && plain_record(info) ? REC_SOLO : REC_GROUP;
    else R.kind = i > 0 && J.pos[q - 1] == pos ? REC_NONE : REC_GROUP;
    return R;
}


static_assert(dense_lds(MAX_BINS, MAX_BITS) + sizeof(count_tables) + DENSE_WAVES * sizeof(slow_list) + TODO_CAP * sizeof(todo) +
                      sizeof(cn_window) + 64 <= 160 * 1024,
              "the widest window (71 KB: mates 4,000 bases away) fits a compute unit's LDS");

template <bool CNA, bool MANY>
__global__ void __launch_bounds__(DENSE_BLOCK, 6) k_count_dense(const seq_launch L) {
    extern __shared__ uint4 s_dyn[];
    __shared__ count_tables s_tab;
    __shared__ uint32_t s_run, s_acc, s_neff, s_todo_n[2];
    using slow_store = std::conditional_t<MANY, slow_list, one_list>;
    __shared__ __align__(16) slow_store s_slow[DENSE_WAVES];  // per wave: a slow template's errors, or those that wait
    __shared__ todo s_todo[TODO_CAP];
    __shared__ cn_window s_cn;  // copy numbers
    uint32_t* const s_bits = (uint32_t*)s_dyn;
    uint32_t* const s_bin = s_bits + L.bit_words;
    uint32_t* const s_cnt = s_bin + L.bins * BIN_STRIDE;  // two sets: one fills while the other is cleared
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    slow_store* const sl = &s_slow[wave];
    uint32_t* const list = sl->list;
    uint32_t in_tab = UNRESOLVED;
    for (uint32_t run = blockIdx.x;;) {
        const item_run R0 = run_of(L, run);
        if (R0.first == R0.end) break;
        if (tid == 0) s_run = gridDim.x + (uint32_t)atomicAdd(L.queue, 1ull);  // the block's next run
        for (uint32_t item = R0.first; item < R0.end; ++item) {
            const item_dev it = uniform_at(L.items, item);
            const seg_dev& S = *(const seg_dev*)((const __attribute__((address_space(4))) seg_dev*)L.segs + it.seg);
            const job_dev& J = *(const job_dev*)((const __attribute__((address_space(4))) job_dev*)L.jobs + S.job);
            const uint32_t c2 = (S.chr << 16) | S.so;
            const uint32_t lns = seg_lns(S), cb = seg_cb(S), lw = seg_lw(S), SH = 32u - lw;
            const uint32_t nslot = DENSE_WAVES >> lns, slot = wave & (nslot - 1u);
            const uint32_t RL = J.L, pe = J.pe, err_n = J.err_n, err_N = J.err_N;
            const source_draw D(J, S, CNA);
            uint32_t errT[4];  // thresholds of 1 to 4 errors past the table's first count (capped below)
#pragma unroll
            for (uint32_t q = 0; q < 4u; ++q) errT[q] = q < err_n ? uniform_at(J.err_T, q) : 0xFFFFFFFFu;
            if (CNA && tid == 0) s_acc = 0;
            if (in_tab != S.job) {
                in_tab = S.job;
                load_count_tables<DENSE_BLOCK>(J, s_tab, tid);
            }
            uint32_t acc = 0;  // accepted templates (copy-number events)
            for (uint32_t jw = it.j0; jw < it.j1; jw += 1u << lns) {
                const uint32_t wb = jw * PSX_STRATUM;
                const uint32_t je = min(jw + (1u << lns), it.j1);
                const uint32_t wend = min(S.len, min(je * PSX_STRATUM, S.W) - 1u + J.reach);
                const uint32_t k0 = uniform_at(J.bucket, S.bucket_off + jw);
                const uint32_t n_win = window_records(J, S, k0, wend);
                // the window's record positions and how many of its records reads can reach
                if (err_n)
                    for (uint32_t i = tid; i < (wend - wb + 31u) >> 5; i += DENSE_BLOCK) s_bits[i] = 0;
                for (uint32_t i = tid; i < L.bins; i += DENSE_BLOCK) s_cnt[i] = 0;
                if (tid == 0) s_neff = s_todo_n[0] = 0;
                if (CNA && S.n_cna && wave == 0) {
                    const uint32_t starts = min(je * PSX_STRATUM, S.W);
                    cn_fill(J, S, wb, starts, lane, s_cn);
                    wave_sync();
                    cn_share(J, S, wb, starts, lane, s_cn);
                }
                __syncthreads();
                for (uint32_t i0 = 0; i0 < n_win; i0 += DENSE_BLOCK) {
                    const uint32_t i = i0 + tid;
                    const uint32_t p = i < n_win ? J.pos[k0 + i] : wend;
                    const bool in = p < wend;
                    if (in && err_n) atomicOr(&s_bits[(p - wb) >> 5], 1u << ((p - wb) & 31u));
                    const uint32_t n = (uint32_t)__popcll(__ballot(in));
                    if (lane == 0 && n) atomicAdd(&s_neff, n);
                }
                __syncthreads();
                const uint32_t n_rec = __builtin_amdgcn_readfirstlane(s_neff);
                // threads per record: the most (up to 32) with all records at once
                uint32_t lgt = 0;
                while (lgt < 5u && (n_rec << (lgt + 1u)) <= DENSE_BLOCK) ++lgt;
                const uint32_t sub = tid & ((1u << lgt) - 1u), step = 1u << lgt;
                const uint32_t per_pass = DENSE_BLOCK >> lgt;
                const bool one_pass = n_rec <= per_pass;
                const uint32_t n_ev = CNA && S.n_cna ? (uint32_t)__builtin_amdgcn_readfirstlane((int)s_cn.n) : CN_GENERAL;
                // the wave's stratum: its templates [t0, t1)
                const uint32_t j = jw + wave / nslot;
                const uint32_t b = j * PSX_STRATUM, e = min(b + PSX_STRATUM, S.W);
                uint32_t t0 = 0, t1 = 0;
                if (j < je) wave_share(S, it.part, b, e, lane, t0, t1);
                // rounds: the same number for every wave, from a bound on any stratum's share
                const uint32_t most = S.most;
                uint32_t round_t = S.round_t;
                if (CNA && S.n_cna) {
                    // of a round's templates only a share has reads: rounds of more templates, as many in each
                    const uint32_t fit = __float2uint_rz(fminf((float)round_t * 1024.0f /
                                                               (float)__builtin_amdgcn_readfirstlane((int)s_cn.share),
                                                               (float)most));
                    const uint32_t rounds = (most + fit - 1u) / max(fit, 1u);
                    round_t = ((most + rounds - 1u) / max(rounds, 1u) + 63u) & ~63u;
                }
                scan_rec R{0, 0, 0, REC_NONE};
                uint32_t dep = 0, alt = 0, set = 0;
                if constexpr (MANY) {
                    if (lane == 0) {
                        sl->n = 0;
                        sl->j = j;
                        sl->c2 = c2;
                        sl->wb = wb;
                        sl->k0 = k0;
                        sl->n_win = n_win;
                        sl->cb = cb;
                        sl->bits = s_bits;
                    }
                }
                for (uint32_t q0 = 0; q0 < most; q0 += round_t) {
                    uint32_t* const cnt = s_cnt + set * L.bins;
                    // ---- draw the round's templates, drop their reads into bins
                    pending P;  // copy numbers: accepted templates
                    const uint32_t end = min(t0 + q0 + round_t, t1);
                    for (uint32_t g = t0 + q0 + slot * 64u;; g += nslot * 64u) {  // wave-uniform
                        const bool more = g < end;
                        bool have = more, on = false;
                        uint32_t x = 0, ins = 0, X = 0, r = g;  // start in the window, insert draw, copy, index
                        if (more) {
                            on = g + lane < end;
                            r = on ? g + lane : g;
                            uint32_t cell, al;
                            const bool ok = D.draw<CNA>(J, S, &s_cn, n_ev, r, j, c2, b, e, wb, x, ins, cell, al);
                            X = (al << cb) | cell;
                            if (CNA) on = on && ok;
                        }
                        if (CNA) {
                            acc += on ? 1u : 0u;
                            have = P.pack(more, on, lane, x, ins, X, r);
                        }
                        uint32_t ev = 0;  // the lane's rare events: full bins (bits 0, 1), errors at records (2, 3, 4)
                        uint32_t P0 = 0, P1 = 0, P2 = 0, subs = 0;
                        unsigned long long slow = 0;
                        const uint32_t d = have ? D.offset(J, s_tab, ins, wb, x) : 0u;
                        if (have) {
                            auto put = [&](uint32_t xr) {  // whether the bin is full
                                const uint32_t bin = xr >> lw;
                                const uint32_t k = atomicAdd(&cnt[bin], 1u);
                                s_bin[__umul24(bin, BIN_STRIDE) + min(k, BIN_CAP)] = (xr << SH) | X;
                                return k >= BIN_CAP;
                            };
                            bool f0 = false, f1 = false;
                            if (on) {
                                f0 = put(x);
                                if (pe) f1 = put(x + d);
                            }
                            if (__ballot(f0 || f1)) ev = (f0 ? 1u : 0u) | (f1 ? 2u : 0u);
                            if (err_n) {
                                // the template's errors (template_errors): all but the slow templates' are settled by
                                // their first draw
                                const psx_u4 w = psx_draw_u(J.seed, r, j, c2, PSX_P_ERROR << 24);
                                uint32_t K = 0;
#pragma unroll
                                for (uint32_t q = 0; q < 4u; ++q) K += w.y >= errT[q] ? 1u : 0u;
                                K = on ? J.err_k0 + min(K, err_n - 1u) : 0u;
                                // position of base bi of the template; whether a record lies there
                                const uint32_t x2 = x + d - RL;
                                auto at = [&](uint32_t bi) { return bi + (bi >= RL ? x2 : x); };
                                auto hit = [&](uint32_t p) { return (s_bits[p >> 5] >> (p & 31u)) & 1u; };
                                const uint32_t b0 = psx_mulhi32(w.x, err_N);
                                const unsigned long long m2 = __ballot(K >= 2u);
                                if (m2) {  // a second and third error; slow templates (any repeated index among b0, b1, b2)
                                    const uint32_t b1 = psx_mulhi32(w.z, err_N), b2 = psx_mulhi32(w.w, err_N);
                                    slow = m2 & (__ballot(K > 3u) | __ballot(b1 == b0) | __ballot(b2 == b0) |
                                                 __ballot(b2 == b1));
                                    if (slow) K = (slow >> lane) & 1ull ? 0u : K;
                                    if (K >= 2u) {
                                        P1 = at(b1);
                                        ev |= hit(P1) << 3;
                                        if (K >= 3u) {
                                            P2 = at(b2);
                                            ev |= hit(P2) << 4;
                                        }
                                    }
                                }
                                if (K >= 1u) {
                                    P0 = at(b0);
                                    ev |= hit(P0) << 2;
                                }
                                if (__ballot(ev > 3u))
                                    subs = (((w.x & 0xFFFFu) * 3u) >> 16) | ((((w.z & 0xFFFFu) * 3u) >> 16) << 2) |
                                           ((((w.w & 0xFFFFu) * 3u) >> 16) << 4);
                            }
                        }
                        // the group's rare events
                        if constexpr (MANY) {
                            if (slow) dense_wait(&J, &S, sl, slow, r, X, x, d);
                            while (__ballot(ev != 0u)) {
                                const bool add = ev != 0u;
                                const uint32_t f = add ? (uint32_t)__ffs((int)ev) - 1u : 0u;
                                ev &= ev - 1u;
                                todo q;
                                q.at = f < 2u ? (x + (f ? d : 0u)) | TODO_READ
                                              : (f == 2u ? P0 : (f == 3u ? P1 : P2)) | ((subs >> (2u * (f - 2u))) & 3u) << 18;
                                q.copy = X;
                                if (add) {
                                    const uint32_t k = atomicAdd(&s_todo_n[set], 1u);
                                    if (k < TODO_CAP) s_todo[k] = q;
                                    else dense_todo(&J, &S, q, wb, k0, n_win, cb);
                                }
                            }
                        } else {
                            uint32_t sl_n = 0, sl_k = 0;  // the current slow template's errors and the next one
                            uint32_t sx = 0, sd = 0, sX = 0;
                            while (__ballot(ev != 0u) || slow || sl_k < sl_n) {
                                bool add = false;
                                todo q{0, 0};
                                if (__ballot(ev != 0u)) {
                                    add = ev != 0u;
                                    const uint32_t f = add ? (uint32_t)__ffs((int)ev) - 1u : 0u;
                                    ev &= ev - 1u;
                                    q.at = f < 2u ? (x + (f ? d : 0u)) | TODO_READ
                                                  : (f == 2u ? P0 : (f == 3u ? P1 : P2)) | ((subs >> (2u * (f - 2u))) & 3u) << 18;
                                    q.copy = X;
                                } else if (sl_k < sl_n) {
                                    const uint32_t k = sl_k + lane;
                                    const uint32_t w = k < sl_n ? list[k] : 0u, bi = w & 0xFFFFFu;
                                    const uint32_t p = bi + (bi >= RL ? sx + sd - RL : sx);
                                    add = k < sl_n && ((s_bits[p >> 5] >> (p & 31u)) & 1u);
                                    q.at = p | (w >> 20) << 18;
                                    q.copy = sX;
                                    sl_k += 64u;
                                } else {  // wave-uniform
                                    const int ln = __ffsll((long long)slow) - 1;
                                    slow &= slow - 1ull;
                                    sx = (uint32_t)__builtin_amdgcn_readlane((int)x, ln);
                                    sd = (uint32_t)__builtin_amdgcn_readlane((int)d, ln);
                                    sX = (uint32_t)__builtin_amdgcn_readlane((int)X, ln);
                                    const uint32_t rs = (uint32_t)__builtin_amdgcn_readlane((int)r, ln);
                                    sl_n = (uint32_t)__builtin_amdgcn_readfirstlane((int)dense_one_slow(&J, rs, j, c2, list));
                                    sl_k = 0;
                                    continue;
                                }
                                if (add) {
                                    const uint32_t k = atomicAdd(&s_todo_n[set], 1u);
                                    if (k < TODO_CAP) s_todo[k] = q;
                                    else dense_todo(&J, &S, q, wb, k0, n_win, cb);
                                }
                            }
                        }
                        if (!more) break;
                    }
                    __syncthreads();
                    // ---- scan: each record's reads among the bins around it
                    const uint32_t n_todo = min(s_todo_n[set], TODO_CAP);
                    if (tid < n_todo) dense_todo(&J, &S, s_todo[tid], wb, k0, n_win, cb);
                    set ^= 1u;
                    for (uint32_t i = tid; i < L.bins; i += DENSE_BLOCK) s_cnt[set * L.bins + i] = 0;
                    if (tid == 0) s_todo_n[set] = 0;
                    const job_dev& Js = reread(J);
                    const seg_dev& Ss = reread(S);
                    for (uint32_t r0 = 0; r0 < n_rec; r0 += per_pass) {
                        const uint32_t i = r0 + (tid >> lgt);
                        if (!one_pass || q0 == 0u)
                            R = i < n_rec ? load_rec(Js, Ss, wb, k0, i, cb, lw) : scan_rec{0, 0, 0, REC_NONE};
                        const int lb = (int)(R.p - (RL - 1u));  // reads over it start at [lb, p]
                        const uint32_t first = R.kind == REC_NONE ? 1u : (uint32_t)max(lb, 0) >> lw;
                        const uint32_t last = R.kind == REC_NONE ? 0u : min(R.p >> lw, L.bins - 1u);
                        for (uint32_t bn = first; bn <= last; ++bn) {
                            const uint32_t n = min(cnt[bn], BIN_CAP);
                            const int at = (int)(bn << lw);
                            const uint32_t plo = (uint32_t)max(lb - at, 0), phi = min(R.p - (uint32_t)at, (1u << lw) - 1u);
                            const uint32_t elo = plo << SH, elen = ((phi - plo + 1u) << SH) - 1u;
                            const uint32_t* const bin = s_bin + bn * BIN_STRIDE;
                            if (R.kind == REC_SOLO) {
                                auto test = [&](uint32_t w) {
                                    const bool over = w - elo <= elen;
                                    dep += over ? 1u : 0u;
                                    alt += over && (w << lw) - R.low < R.len ? 1u : 0u;
                                };
                                for (uint32_t k = sub; k < n >> 2; k += step) {
                                    const uint4 w = ((const uint4*)bin)[k];
                                    test(w.x);
                                    test(w.y);
                                    test(w.z);
                                    test(w.w);
                                }
                                for (uint32_t k = (n & ~3u) + sub; k < n; k += step) test(bin[k]);
                            } else {
                                dense_group(&J, &S, bin, sub, n, step, elo, elen, lw, cb, k0, n_win, i);
                            }
                        }
                        if (!one_pass || q0 + round_t >= most) {
                            for (uint32_t m = 1; m < step; m <<= 1) {
                                dep += (uint32_t)__shfl_xor((int)dep, (int)m);
                                alt += (uint32_t)__shfl_xor((int)alt, (int)m);
                            }
                            if (sub == 0u && dep) {
                                const uint64_t o = out_off(Js, Ss) + k0 + i;
                                atomicAdd(Js.depth + o, (int32_t)dep);
                                if (alt) atomicAdd(Js.alt + o, (int32_t)alt);
                            }
                            dep = alt = 0;
                        }
                    }
                    __syncthreads();
                }
                if constexpr (MANY) {
                    if (__builtin_amdgcn_readfirstlane((int)sl->n)) dense_slow(&J, &S, sl);
                }
                __syncthreads();
            }
            if (CNA && S.n_cna) {
                if (acc) atomicAdd(&s_acc, acc);
                __syncthreads();
                if (tid == 0 && s_acc) atomicAdd(J.acc, (unsigned long long)s_acc * (J.pe + 1u));
                __syncthreads();
            }
        }
        __syncthreads();
        run = __builtin_amdgcn_readfirstlane(s_run);
        __syncthreads();  // read by every wave before it is written again
    }
}

}  // namespace psxk
