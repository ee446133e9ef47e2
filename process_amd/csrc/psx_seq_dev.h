// Device side of simulate_seq on gfx950: descriptors, the draws of templates
// and their errors, and the read-materialising kernel (the count-only kernels:
// psx_count_dev.h). Included once, by psx_seq.hip.
//
// Work decomposition. A segment is one (job, output sample, chromosome); its
// W = len - L + 1 template starts are cut into strata of PSX_STRATUM starts,
// and stratum j owns a fixed number of templates (part of the sampling model,
// so results do not depend on the launch). A work item is a run of strata of
// one segment; persistent blocks pull runs of items from a device counter.
//
// Per stratum the read kernel stages in LDS the SNVs that the stratum's reads
// can carry, with a 32-base bucket index, the reference under them and the job's
// inversion tables; reads are generated from counters and built from there.
#pragma once
#include "psx_cna.h"
#include "psx_internal.h"

namespace psxk {

constexpr uint32_t NB_SHIFT = 5;      // 32-base LDS buckets
constexpr uint32_t MAX_READ = 4096;   // read size and insert reach limit
constexpr uint32_t NB_MAX = ((PSX_STRATUM + MAX_READ) >> NB_SHIFT) + 2;
constexpr uint32_t MAX_INS = 640;     // compact insert-size thresholds in LDS
constexpr uint32_t MAX_ERRT = PSX_ERR_KCAP + 1;
constexpr uint32_t REF_MAX = (PSX_STRATUM + MAX_READ) / 16 + 4;
constexpr uint32_t UNRESOLVED = 0xFFFFFFFFu;

// Descriptors are read-only for the whole launch: reading them through the
// constant address space lets the compiler use scalar loads, so the fields
// live in SGPRs instead of taking VGPRs from every lane.
template <class T>
__device__ __forceinline__ T uniform_at(const T* p, uint64_t i) {
#if defined(__HIP_DEVICE_COMPILE__)
    return ((const __attribute__((address_space(4))) T*)p)[i];
#else
    return p[i];
#endif
}

struct job_dev {
    uint64_t seed;
    const uint32_t* pos;
    const uint32_t* lo;
    const uint32_t* hi;
    const uint32_t* info;
    const uint32_t* bucket;
    const uint32_t* sample_leaves;
    const uint4* leaf_count;     // per sample and 64 leaf ranks: {leaves below, membership bits, 0}
    int32_t* alt;
    int32_t* depth;
    uint8_t* present;
    const uint32_t* ins_T;       // compact insert-size thresholds
    const uint16_t* ins_guide;
    const uint32_t* err_T;       // compact thresholds of the errors per template
    const uint32_t* packed;      // reference (read materialisation)
    uint64_t n_mut;
    uint64_t thr_normal;         // floor((1 - purity) 2^32)
    uint32_t ins_k0, ins_n;
    uint32_t err_n, err_k0;      // error table (err_n == 0: no sequencing errors)
    uint32_t err_N;              // bases per template: (pe + 1) L
    uint32_t pad;                // the fields from here on start at 16 bytes: without it every small count takes 0.5-1 % longer
    uint32_t L, pe, ploidy, n_leaves, preneo, reach;
    uint32_t n_out;
    uint32_t purity_lt1;
    uint32_t leaf_blocks;        // leaf_count entries per sample
    const psx_cna_dev* cna;      // copy-number events of every chromosome, per segment ranges
    unsigned long long* acc;     // reads of accepted templates (jobs with copy-number events)
    const uint64_t* cn_row;      // read materialisation: first read of each copy-number stratum (seg st_off + j)
};

struct seg_dev {
    uint64_t T;             // templates of the segment
    uint32_t sample;        // the forest sample (tumour samples)
    uint32_t shape;         // seg_parts << 16, and for the count kernels seg_cb | seg_lns << 8 | seg_lw << 12
    union {
        uint64_t read_base;  // materialisation: first read index of the segment
        struct {             // dense count kernel: most templates of an item's part of a stratum, and of a round of it
            uint32_t most, round_t;
        };
    };
    uint64_t chr_woff;      // first packed word of the chromosome
    uint32_t job, so, chr, len;
    uint32_t W, J, bucket_off;
    uint32_t spi;                // strata per work item
    uint32_t leaf_off, n_cells;  // n_cells == 0: normal sample
    uint32_t cna_off, n_cna;     // the chromosome's copy-number events (J.cna + cna_off)
    uint32_t kmax;               // copies drawn per template: the largest copy number, >= ploidy
    uint32_t first_item;         // its work items: first_item .. first_item + ceil(J / spi) seg_parts - 1
    uint32_t st_off;             // segments with copy-number events: index of its first stratum in J.cn_row
};

// Bits of a cell index of the segment's sample (its number of cells included); log2 of the strata of a window of the
// dense count kernel and of the starts of its bins; the parts each item's templates are cut into (items of few strata
// with many templates).
__host__ __device__ __forceinline__ uint32_t seg_cb(const seg_dev& S) { return S.shape & 0xFFu; }
__host__ __device__ __forceinline__ uint32_t seg_lns(const seg_dev& S) { return (S.shape >> 8) & 0xFu; }
__host__ __device__ __forceinline__ uint32_t seg_lw(const seg_dev& S) { return (S.shape >> 12) & 0xFu; }
__host__ __device__ __forceinline__ uint32_t seg_parts(const seg_dev& S) { return S.shape >> 16; }

struct item_dev {
    uint32_t seg, j0, j1, part;
};

// The work items of a batch, written on the device from the segments (the
// host lists segments only): item q belongs to the last segment whose first
// item is at or below q (a segment without templates has no items and shares
// its successor's first item) and covers its part of spi strata from its first.
__global__ void __launch_bounds__(256) k_seq_items(const seg_dev* __restrict__ segs, uint32_t n_segs,
                                                   item_dev* __restrict__ items, uint32_t n_items) {
    const uint32_t q = blockIdx.x * 256u + threadIdx.x;
    if (q >= n_items) return;
    uint32_t a = 0, z = n_segs;
    while (a < z) {
        const uint32_t mid = (a + z) >> 1;
        if (segs[mid].first_item <= q) a = mid + 1; else z = mid;
    }
    const seg_dev& S = segs[a - 1];
    const uint32_t run = (q - S.first_item) / seg_parts(S), part = (q - S.first_item) - run * seg_parts(S);
    const uint32_t j0 = run * S.spi;
    items[q] = item_dev{a - 1, j0, min(S.J, j0 + S.spi), part};
}

struct pres_dev {  // one per (job, output sample) for the init kernel
    uint64_t begin;        // global index of the first (so, m) entry
    uint32_t job, so, leaf_off, n_cells;
    uint32_t sample, pad;  // the forest sample of the output sample (tumour samples)
};

struct seq_launch {
    const job_dev* jobs;
    const seg_dev* segs;
    const item_dev* items;
    uint64_t n_items;
    unsigned long long* queue;
    uint32_t chunk;          // items taken at a time (run_of)
    uint32_t bins;           // dense count kernel: bins of a window, words of its position bitmap
    uint32_t bit_words;
    uint32_t* reads_out;     // materialisation only
    uint32_t read_words;
    uint32_t out_vec4;       // read_words % 4 == 0 and reads_out 16-byte aligned
    const uint64_t* cn_kept; // segments with copy-number events: which templates are kept (cn_groups words a stratum)
};

// The items of a persistent launch are handed out in runs of L.chunk: block b
// takes run b without asking, later ones from the counter. Atomics on the one
// counter serialise at about 12 ns each whatever the items hold, which set the
// time of every launch of many small items (147,000 strata of a 10x run: 1.79
// ms, of which the counter 1.76); in runs of about 8,192 templates the counter
// costs 1.5 ps per template against the kernels' 5-11.
struct item_run {
    uint32_t first, end;
};
__device__ __forceinline__ item_run run_of(const seq_launch& L, uint32_t run) {
    const uint64_t first = (uint64_t)run * L.chunk;
    if (first >= L.n_items) return item_run{0u, 0u};
    const uint64_t left = L.n_items - first;
    return item_run{(uint32_t)first, (uint32_t)(first + (left < L.chunk ? left : L.chunk))};
}

// The job's inversion tables in LDS (the read kernel's; the count kernels': count_tables).
struct lds_tables {
    uint32_t ins[MAX_INS];
    uint16_t guide[PSX_GUIDE];
    uint32_t err[MAX_ERRT];
};

__device__ __forceinline__ void load_tables(const job_dev& J, lds_tables& t, uint32_t tid, uint32_t block) {
    if (J.pe) {
        for (uint32_t i = tid; i < J.ins_n; i += block) t.ins[i] = J.ins_T[i];
        for (uint32_t i = tid; i < PSX_GUIDE; i += block) t.guide[i] = J.ins_guide[i];
    }
    for (uint32_t i = tid; i < J.err_n; i += block) t.err[i] = J.err_T[i];
    // the error-count pick reads thresholds 0..3 whatever the table's length
    for (uint32_t i = J.err_n + tid; i < 4u; i += block) t.err[i] = 0xFFFFFFFFu;
}

// LDS writes of a wave visible to its other lanes.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ------------------------------------------------------------- record views

struct lds_view {  // the read kernel's staged records
    const uint32_t* pos;
    const uint32_t* lo;
    const uint32_t* hi;
    const uint32_t* info;
    const uint16_t* bucket;
    uint32_t n, b;
    // a record index at or before the first record at or after x
    __device__ __forceinline__ uint32_t start(uint32_t x) const { return bucket[(x - b) >> NB_SHIFT]; }
    __device__ __forceinline__ uint32_t at(uint32_t i) const { return min(i, n - 1u); }  // n > 0
};

struct glb_view {  // records in global memory
    const uint32_t* pos;
    const uint32_t* lo;
    const uint32_t* hi;
    const uint32_t* info;
    int32_t* alt;
    int32_t* dep;
    uint32_t n;
    __device__ __forceinline__ uint32_t first(uint32_t x) const {
        uint32_t a = 0, z = n;
        while (a < z) {
            const uint32_t mid = (a + z) >> 1;
            if (pos[mid] < x) a = mid + 1; else z = mid;
        }
        return a;
    }
    __device__ __forceinline__ uint32_t start(uint32_t x) const { return first(x); }
    __device__ __forceinline__ uint32_t at(uint32_t i) const { return min(i, n - 1u); }  // n > 0
    __device__ __forceinline__ void add_dep(uint32_t q) const { atomicAdd(&dep[q], 1); }
    __device__ __forceinline__ void add_alt(uint32_t q) const { atomicAdd(&alt[q], 1); }
    __device__ __forceinline__ void add_alt_n(uint32_t q, int d) const { atomicAdd(&alt[q], d); }
};

// Template: start of mate 1 and mate 2, source cell and its leaf, and copy;
// ok == 0 when a copy-number draw rejects it.
struct tmpl {
    uint32_t x, x2, cell, allele, leaf, ok;
};

// Copy numbers of a leaf at base x of the segment's chromosome, from its
// events read with scalar loads (the list is the same for every lane);
// returns the total. Oracle: copies.
__device__ __forceinline__ uint32_t cna_copies(const psx_cna_dev* ev, uint32_t n, uint32_t leaf, uint32_t x,
                                               uint32_t ploidy, uint32_t* cn) {
#pragma unroll
    for (uint32_t a = 0; a < PSX_MAX_CNA_PLOIDY; ++a) cn[a] = a < ploidy ? 1u : 0u;
    for (uint32_t i = 0; i < n; ++i) {
        const psx_cna_dev e = uniform_at(ev, i);
        const bool hit = leaf >= e.lo && leaf < e.hi && x >= e.start && x < e.end;
        const uint32_t a = e.code & 0xFFu, kind = (e.code >> 8) & 0xFFu, c = e.code >> 16;
#pragma unroll
        for (uint32_t q = 0; q < PSX_MAX_CNA_PLOIDY; ++q) {
            const uint32_t v = cn[q];
            const uint32_t nv = kind == PSX_CNA_WGD ? 2u * v : (q != a ? v : (kind == PSX_CNA_AMP ? v + c : 0u));
            cn[q] = hit ? nv : v;
        }
    }
    uint32_t total = 0;
#pragma unroll
    for (uint32_t a = 0; a < PSX_MAX_CNA_PLOIDY; ++a) total += cn[a];
    return total;
}

// cna_copies of a diploid leaf: the copies of its two lineages. The event is the same for every lane, so its kind is a
// uniform branch, and the next one is read meanwhile: bound by vector instruction issue, 7 instructions an event where
// the walk for any ploidy takes 30. Windows under 17 events (60x pairs of 150 bases over 17.5 Mb): 1,328 -> 690 us
// counted, 2,650 -> 1,810 a call that materialises 20x.
__device__ __forceinline__ void cna_copies2(const psx_cna_dev* ev, uint32_t n, uint32_t leaf, uint32_t x, uint32_t& c0,
                                            uint32_t& c1) {
    c0 = c1 = 1u;
    if (n == 0u) return;
    psx_cna_dev e = uniform_at(ev, 0);
    for (uint32_t i = 0; i < n; ++i) {
        const psx_cna_dev next = uniform_at(ev, min(i + 1u, n - 1u));
        const bool hit = (leaf - e.lo < e.hi - e.lo) & (x - e.start < e.end - e.start);
        const uint32_t a = e.code & 0xFFu, kind = (e.code >> 8) & 0xFFu, c = e.code >> 16;
        if (kind == PSX_CNA_WGD) {
            c0 = hit ? 2u * c0 : c0;
            c1 = hit ? 2u * c1 : c1;
        } else if (a == 0u) {
            c0 = hit ? (kind == PSX_CNA_AMP ? c0 + c : 0u) : c0;
        } else {
            c1 = hit ? (kind == PSX_CNA_AMP ? c1 + c : 0u) : c1;
        }
        e = next;
    }
}

// Cells of the sample with leaf ranks below x, from the sample's running counts.
__device__ __forceinline__ uint32_t cells_below(const job_dev& J, uint32_t sample, uint32_t x) {
    const uint4 e = J.leaf_count[(uint64_t)sample * J.leaf_blocks + (x >> 6)];
    const uint64_t bits = (uint64_t)e.y | ((uint64_t)e.z << 32);
    return e.x + (uint32_t)__popcll(bits & ((1ull << (x & 63u)) - 1ull));
}

// The copy-number events of a diploid segment that touch a window of starts,
// with their leaf ranges as ranges of the sample's cells: [cell, cell + cells),
// [start, start + starts), and what they do to the packed copies of the two
// lineages, ((C & keep) << twice) + add. A template needs no look-up of its
// leaf and no division, and walks the events of its window alone, in LDS: the
// counts of 3.3e8 templates of 9e8 draws (500x, 13 events on 10 chromosomes)
// 4.8 -> 4.1 ms. Bound by vector instruction issue: 173 instructions a group of
// 64 draws with the reads queued, 43 of them Philox.
struct cn_event {
    uint32_t cell, cells, start, starts;
    uint32_t keep, twice, add, pad;
};
constexpr uint32_t CN_EVENTS = 16;
constexpr uint32_t CN_DOUBLINGS = 3;  // an event adds at most 255: (1 + 16 * 255) << 3 < 2^16, no lineage overflows its half
struct cn_window {
    cn_event ev[CN_EVENTS];
    uint32_t n;
    uint32_t share;  // about the largest share of the templates, of any quarter of the window, that is kept, times 2^10
};
constexpr uint32_t CN_GENERAL = 0xFFFFFFFFu;  // not in this form: drawn by template_source

// One wave fills w with the events of S that touch the starts [b, e).
__device__ __forceinline__ void cn_fill(const job_dev& J, const seg_dev& S, uint32_t b, uint32_t e, uint32_t lane,
                                        cn_window& w) {
    uint32_t n = 0, doubled = 0;
    const bool general = J.ploidy != 2u;
    for (uint32_t i0 = 0; S.n_cells && i0 < S.n_cna; i0 += 64u) {
        const uint32_t i = i0 + lane;
        cn_event q{};
        uint32_t kind = 0;
        bool on = i < S.n_cna;
        if (on) {
            const psx_cna_dev d = J.cna[S.cna_off + i];
            const uint32_t a = d.code & 0xFFu;
            kind = (d.code >> 8) & 0xFFu;
            const uint32_t c = kind == PSX_CNA_AMP ? d.code >> 16 : 0u;
            q.cell = cells_below(J, S.sample, d.lo);
            q.cells = cells_below(J, S.sample, d.hi) - q.cell;
            q.start = d.start;
            q.starts = d.end - d.start;
            q.keep = kind == PSX_CNA_DEL ? (a == 0u ? 0xFFFF0000u : 0xFFFFu) : 0xFFFFFFFFu;
            q.twice = kind == PSX_CNA_WGD ? 1u : 0u;
            q.add = a == 0u ? c : c << 16;
            on = d.start < e && d.end > b && q.cells != 0u;
        }
        const unsigned long long m = __ballot(on);
        const uint32_t at = n + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
        if (on && at < CN_EVENTS) w.ev[at] = q;
        n += (uint32_t)__popcll(m);
        doubled += (uint32_t)__popcll(__ballot(on && kind == PSX_CNA_WGD));
    }
    if (lane == 0) w.n = general || n > CN_EVENTS || doubled > CN_DOUBLINGS ? CN_GENERAL : n;
}

// The packed copies of a cell at start x.
__device__ __forceinline__ uint32_t cn_copies(const cn_window& w, uint32_t n_ev, uint32_t cell, uint32_t x) {
    uint32_t C = 0x10001u;  // lineage 0 | lineage 1 << 16
    for (uint32_t i = 0; i < n_ev; ++i) {
        const cn_event& q = w.ev[i];
        const bool hit = (cell - q.cell < q.cells) & (x - q.start < q.starts);
        const uint32_t D = ((C & q.keep) << q.twice) + q.add;
        C = hit ? D : C;
    }
    return C;
}

// The share of templates kept, by one wave after cn_fill: 64 cells in the
// middle of each quarter of the window. It only sizes the rounds.
__device__ __forceinline__ void cn_share(const job_dev& J, const seg_dev& S, uint32_t b, uint32_t e, uint32_t lane,
                                         cn_window& w) {
    const uint32_t n_ev = (uint32_t)__builtin_amdgcn_readfirstlane((int)w.n);
    float most = 0.0f;
    for (uint32_t q = 0; n_ev != CN_GENERAL && q < 4u; ++q) {
        const uint32_t C = cn_copies(w, n_ev, (uint32_t)(((uint64_t)S.n_cells * (2u * lane + 1u)) >> 7),
                                     b + (uint32_t)(((uint64_t)(e - b) * (2u * q + 1u)) >> 3));
        float sum = (float)((C & 0xFFFFu) + (C >> 16));
        for (uint32_t m = 1; m < 64u; m <<= 1) sum += __shfl_xor(sum, (int)m);
        most = fmaxf(most, sum);
    }
    const float normal = S.n_cells ? (float)J.thr_normal * 0x1p-32f : 1.0f;
    const float kept = n_ev == CN_GENERAL ? 1.0f : ((1.0f - normal) * most * 0x1p-6f + normal * 2.0f) / (float)S.kmax;
    if (lane == 0) w.share = (uint32_t)fminf(fmaxf(kept, 0x1p-6f) * 1024.0f, 1024.0f);
}

// The source of a template that starts at x, from word z of its draw: cell
// (n_cells: the normal genome) and lineage; whether the drawn slot is one of
// its copies. The slot X = floor(z cells K / 2^32) belongs to cell
// floor(X / K) = floor(z cells / 2^32). normal: a tumour sample's template is
// the normal genome's.
__device__ __forceinline__ bool cn_source(const seg_dev& S, const cn_window& w, uint32_t n_ev, bool normal, uint32_t z,
                                          uint32_t x, uint32_t& cell, uint32_t& al) {
    const uint32_t K = S.kmax, n = S.n_cells;
    cell = n;
    if (n == 0u) {  // the normal sample (the same branch for every lane)
        al = psx_uniform32(z, K);
        return al < 2u;
    }
    const uint32_t c = psx_uniform32(z, normal ? 1u : n);
    const uint32_t k = psx_uniform32(z, normal ? K : n * K) - c * K;
    cell = normal ? n : c;
    const uint32_t C = cn_copies(w, n_ev, cell, x);
    const uint32_t c0 = C & 0xFFFFu;
    al = k >= c0 ? 1u : 0u;
    return k < c0 + (C >> 16);
}

__device__ __forceinline__ uint32_t leaf_of(const job_dev& J, const seg_dev& S, tmpl& t) {
    if (t.leaf == UNRESOLVED) t.leaf = J.sample_leaves[S.leaf_off + t.cell];
    return t.leaf;
}

__device__ __forceinline__ bool carried(const job_dev& J, uint32_t info, uint32_t lo, uint32_t hi, uint32_t leaf) {
    if (leaf == J.n_leaves) {
        const uint32_t nat = PSX_INFO_NATURE(info);
        return nat == PSX_GERMINAL || (nat == PSX_PRENEOPLASTIC && J.preneo);
    }
    return lo <= leaf && leaf < hi;
}

// psx_guided_pick with a wave-uniform binary search inside the guide bucket:
// the answer lies in [guide[g], guide[g + 1]] (the last bucket ends at n - 1),
// and the tail buckets of a peaked distribution hold tens of entries, which a
// linear scan would walk for the whole wave. Same result as psx_guided_pick.
__device__ __forceinline__ uint32_t guided_pick_u(const uint32_t* T32, const uint16_t* guide, uint32_t n, uint32_t u) {
    const uint32_t g = u >> (32u - PSX_GUIDE_BITS);
    uint32_t lo = guide[g];
    uint32_t hi = g < PSX_GUIDE - 1u ? guide[g + 1u] : n - 1u;
    while (__ballot(lo < hi)) {
        const uint32_t mid = (lo + hi) >> 1;
        const bool below = u < T32[mid];
        const bool on = lo < hi;
        hi = on && below ? mid : hi;
        lo = on && !below ? mid + 1u : lo;
    }
    return lo;
}

// Template r of stratum j without its mate (oracle: template_source): start,
// source and, with copy-number events, whether the template is kept; without
// LEAF and events the source's leaf is left out. w gets the template draw
// (its word w is the insert size).
template <bool CNA = false, bool LEAF = true>
__device__ __forceinline__ tmpl template_source(const job_dev& J, const seg_dev& S, uint32_t r, uint32_t j,
                                                uint32_t b, uint32_t e, psx_u4& w) {
    const uint32_t c2 = (S.chr << 16) | S.so;
    w = psx_draw_u(J.seed, r, j, c2, PSX_P_TEMPLATE << 24);
    tmpl t;
    t.x = b + psx_uniform32(w.x, e - b);
    t.ok = 1u;
    if (!CNA || S.n_cna == 0) {
        // a copy of a cell, or of the normal genome (cell n_cells)
        const bool normal = S.n_cells == 0 || (uint64_t)w.y < J.thr_normal;
        const uint32_t X = psx_uniform32(w.z, normal ? J.ploidy : S.n_cells * J.ploidy);
        t.cell = normal ? 0u : psx_uniform32(w.z, S.n_cells);  // floor(X / ploidy)
        t.allele = X - t.cell * J.ploidy;
        if (LEAF) {
            t.leaf = J.n_leaves;
            if (!normal) t.leaf = J.sample_leaves[S.leaf_off + t.cell];  // issued early: its latency overlaps the draws
        }
        t.cell = normal ? S.n_cells : t.cell;
    } else {
        // one of kmax copy slots per cell; the template is kept when the slot
        // is one of the source's copies at x, whose lineage it then reads
        const uint32_t K = S.kmax;
        if (S.n_cells == 0 || (uint64_t)w.y < J.thr_normal) {
            const uint32_t k = psx_uniform32(w.z, K);
            t.leaf = J.n_leaves;
            t.cell = S.n_cells;
            t.allele = k;
            t.ok = k < J.ploidy;
        } else {
            t.cell = psx_uniform32(w.z, S.n_cells);  // floor(floor(z cells K / 2^32) / K)
            const uint32_t k = psx_uniform32(w.z, S.n_cells * K) - t.cell * K;
            t.leaf = J.sample_leaves[S.leaf_off + t.cell];
            if (J.ploidy == 2u) {
                uint32_t c0, c1;
                cna_copies2(J.cna + S.cna_off, S.n_cna, t.leaf, t.x, c0, c1);
                t.allele = k >= c0 ? 1u : 0u;
                t.ok = k < c0 + c1;
            } else {
                uint32_t cn[PSX_MAX_CNA_PLOIDY];
                const uint32_t C = cna_copies(J.cna + S.cna_off, S.n_cna, t.leaf, t.x, J.ploidy, cn);
                uint32_t cum = 0, al = 0;
#pragma unroll
                for (uint32_t a = 0; a < PSX_MAX_CNA_PLOIDY; ++a) {
                    cum += cn[a];
                    al += (a + 1 < J.ploidy && k >= cum) ? 1u : 0u;
                }
                t.allele = al;
                t.ok = k < C;
            }
        }
    }
    t.x2 = t.x;
    return t;
}

// Start of mate 2 of a template that starts at x, from the insert word of its draw.
__device__ __forceinline__ uint32_t mate_start(const job_dev& J, const seg_dev& S, const lds_tables& tab, uint32_t x,
                                               uint32_t ins) {
    if (!J.pe) return x;
    uint32_t I = J.ins_k0 + guided_pick_u(tab.ins, tab.guide, J.ins_n, ins);
    if (I < J.L) I = J.L;
    const uint64_t x2 = (uint64_t)x + I - J.L;
    return x2 > S.len - J.L ? S.len - J.L : (uint32_t)x2;
}

// Template r of stratum j of a segment without copy-number events (oracle:
// the template loop of orc_simulate_seq).
__device__ __forceinline__ tmpl make_template(const job_dev& J, const seg_dev& S, const lds_tables& tab, uint32_t r,
                                              uint32_t j, uint32_t b, uint32_t e) {
    psx_u4 w;
    tmpl t = template_source(J, S, r, j, b, e, w);
    t.x2 = mate_start(J, S, tab, t.x, w.w);
    return t;
}

// Templates that start below x: floor(T x / W) (T W < 2^64, x <= W) by a
// double quotient and its exact remainder; a 64-bit integer division is over
// a hundred instructions.
__device__ __forceinline__ uint64_t templates_below(const seg_dev& S, uint32_t x) {
    const uint64_t n = S.T * x, W = S.W;
    uint64_t q = (uint64_t)((double)n / (double)W);
    int64_t r = (int64_t)(n - q * W);
    while (r < 0) {
        --q;
        r += (int64_t)W;
    }
    while (r >= (int64_t)W) {
        ++q;
        r -= (int64_t)W;
    }
    return q;
}

// Whether template r of stratum [b, e) is kept and its draw, start, cell and
// lineage; a segment with copy-number events.
__device__ __forceinline__ bool cn_template(const job_dev& J, const seg_dev& S, const cn_window& cw, uint32_t n_ev,
                                            uint32_t r, uint32_t j, uint32_t b, uint32_t e, psx_u4& w, tmpl& t) {
    if (n_ev == CN_GENERAL) {
        t = template_source<true, false>(J, S, r, j, b, e, w);
        return t.ok != 0u;
    }
    w = psx_draw_u(J.seed, r, j, (S.chr << 16) | S.so, PSX_P_TEMPLATE << 24);
    t.x = b + psx_uniform32(w.x, e - b);
    return cn_source(S, cw, n_ev, (uint64_t)w.y < J.thr_normal, w.z, t.x, t.cell, t.allele);
}

// Groups of 64 templates of a segment's strata (the largest of them).
__device__ __forceinline__ uint32_t cn_groups(const seg_dev& S) {
    return (uint32_t)((templates_below(S, min(PSX_STRATUM, S.W)) + 64u) >> 6);
}
constexpr uint32_t CN_CHUNK = 256;  // groups whose kept templates a block of the read kernel numbers at a time

// Position of set bit n of m (n < the number of set bits).
__device__ __forceinline__ uint32_t nth_set(uint64_t m, uint32_t n) {
    uint32_t w = (uint32_t)m, at = 0;
    const uint32_t c = (uint32_t)__popc(w);
    if (n >= c) { n -= c; w = (uint32_t)(m >> 32); at = 32; }
#pragma unroll
    for (uint32_t s = 16; s; s >>= 1) {
        const uint32_t k = (uint32_t)__popc(w & ((1u << s) - 1u));
        const bool up = n >= k;
        n -= up ? k : 0u;
        w >>= up ? s : 0u;
        at += up ? s : 0u;
    }
    return at;
}

// Sequencing errors of a template (oracle: template_errors). Most templates
// are settled by their first draw w_0: K <= 3 and the stream words x, z, w of
// w_0 give distinct base indices; their errors travel in a two-word summary,
// each error as e = b | sub << 13 (b < 2 L <= 8192 the template's base
// index, sub the substitution index). The others (slow) are generated by the
// whole wave (wave_template_errors).
struct terr {
    uint32_t w01;  // e_0 | e_1 << 16
    uint32_t w2n;  // e_2 | n << 16 | slow << 18
    __device__ __forceinline__ uint32_t n() const { return (w2n >> 16) & 3u; }
    __device__ __forceinline__ bool slow() const { return (w2n >> 18) & 1u; }
};

// The summary of template r of stratum j; lanes with want == false get none.
// Every lane steps through the same count loop.
// err: the error table's first four thresholds (padded).
__device__ __forceinline__ terr template_errors(const job_dev& J, uint64_t seed, const uint32_t* err, uint32_t r,
                                                uint32_t j, uint32_t c2, bool want) {
    const psx_u4 w = psx_draw_u(seed, r, j, c2, PSX_P_ERROR << 24);
    // K = err_k0 + the number of thresholds k < err_n - 1 with u >= T[k] (T is
    // non-decreasing, every kept threshold but the last below 2^32, the last and
    // the padding 2^32 - 1); only K <= 3 matters here, so four compares against
    // the first thresholds (read by every lane alike) give min(K, 4) without a
    // loop, and capping at err_n - 1 drops the last threshold and the padding,
    // which only u = 2^32 - 1 reaches
    uint32_t k = 0;
#pragma unroll
    for (uint32_t q = 0; q < 4u; ++q) k += w.y >= err[q] ? 1u : 0u;
    k = min(k, J.err_n ? J.err_n - 1u : 0u);
    const uint32_t K = want ? J.err_k0 + k : 0u;
    const uint32_t b0 = psx_mulhi32(w.x, J.err_N), b1 = psx_mulhi32(w.z, J.err_N), b2 = psx_mulhi32(w.w, J.err_N);
    const bool slow = K > 3u || (K >= 2u && b1 == b0) || (K >= 3u && (b2 == b0 || b2 == b1));
    const uint32_t n = slow ? 0u : K;
    const uint32_t e0 = b0 | ((((w.x & 0xFFFFu) * 3u) >> 16) << 13);
    const uint32_t e1 = b1 | ((((w.z & 0xFFFFu) * 3u) >> 16) << 13);
    const uint32_t e2 = b2 | ((((w.w & 0xFFFFu) * 3u) >> 16) << 13);
    terr e;
    e.w01 = (n > 0u ? e0 : 0u) | ((n > 1u ? e1 : 0u) << 16);
    e.w2n = (n > 2u ? e2 : 0u) | (n << 16) | ((slow ? 1u : 0u) << 18);
    return e;
}

__device__ __forceinline__ terr shfl_terr(const terr& e, uint32_t src) {
    return terr{(uint32_t)__shfl((int)e.w01, (int)src), (uint32_t)__shfl((int)e.w2n, (int)src)};
}

// The observed base at template base index b whose true base is tb, with the
// summary's errors (none for a slow template).
__device__ __forceinline__ uint32_t observe(const terr& e, uint32_t b, uint32_t tb) {
    const uint32_t n = e.n();
    const uint32_t e0 = e.w01 & 0xFFFFu, e1 = e.w01 >> 16, e2 = e.w2n & 0xFFFFu;
    uint32_t sub = 4u;
    sub = n > 0u && (e0 & 0x1FFFu) == b ? e0 >> 13 : sub;
    sub = n > 1u && (e1 & 0x1FFFu) == b ? e1 >> 13 : sub;
    sub = n > 2u && (e2 & 0x1FFFu) == b ? e2 >> 13 : sub;
    return sub == 4u ? tb : (sub < tb ? sub : sub + 1u);
}

// Per-wave LDS of a slow template's errors: the list, then a 2048-bit hashed
// bitmap of the base indices drawn so far.
constexpr uint32_t ELIST = PSX_ERR_KCAP + 64u;

// All errors of template r (oracle: template_errors), generated by one wave:
// the count K from word y of w_0 (a parallel compare against the
// thresholds), then the stream words in batches, lane l drawing stream word
// t0 + l (x, z, w of w_0, then the four words of w_1, w_2, ...). A word is new
// when no earlier stream word gives the same base index (an earlier equal
// index was taken or was itself a repeat of a taken one), and the first K new
// words are the errors. Repeats are rare: the bitmap flags the lanes that may
// be one, and only such a batch runs the exact check: of every index, or with
// FLAGGED of the flagged lanes' (tens of errors flag a lane of most batches: 7e6
// reads of 1,000 bases at 5 %, counted, 9.5 -> 4.7 ms; the read kernel, whose
// registers are few, keeps the other: 5e7 single-end reads of 100 bases 610 us,
// 625 with FLAGGED). Writes the errors to
// list[0 .. K) as b | sub << 20 and returns K (wave-uniform); every lane
// steps through the same loops. known: K, if the caller has it (above 0).
template <bool FLAGGED = false>
__device__ __forceinline__ uint32_t wave_template_errors(uint64_t seed, uint32_t err_n, uint32_t err_k0, uint32_t err_N,
                                                      const uint32_t* err_T, uint32_t r, uint32_t j, uint32_t c2,
                                                      uint32_t* list, uint32_t lane, uint32_t known = UNRESOLVED) {
    constexpr uint32_t TMAX = 4u * PSX_ERR_KCAP;  // stream words available
    uint32_t* bits = list + PSX_ERR_KCAP;
    uint32_t K = 0, cnt = 0;
    for (uint32_t t0 = 0; t0 < TMAX;) {
        const uint32_t t = t0 + lane;
        const uint32_t call = t < 3u ? 0u : 1u + ((t - 3u) >> 2);
        const psx_u4 w = psx_draw_u(seed, r, j, c2, (PSX_P_ERROR << 24) | call);
        const uint32_t word = psx_word(w, t < 3u ? (t == 0u ? 0 : (int)t + 1) : (int)((t - 3u) & 3u));
        if (t0 == 0 && known != UNRESOLVED) {
            K = known;
            bits[lane] = 0u;
            wave_sync();
        } else if (t0 == 0) {
            // K - err_k0 = the number of thresholds k < err_n - 1 with u >= T[k]
            const uint32_t u = (uint32_t)__builtin_amdgcn_readfirstlane((int)w.y);  // lane 0 drew w_0
            uint32_t k = 0;
            for (uint32_t i0 = 0; i0 + 1u < err_n; i0 += 64u) {
                const uint32_t i = i0 + lane;
                k += (uint32_t)__popcll(__ballot(i + 1u < err_n && u >= err_T[min(i, err_n - 1u)]));
            }
            K = err_k0 + k;
            if (K == 0) return 0;
            bits[lane] = 0u;
            wave_sync();
        }
        const uint32_t B = min(64u, K - cnt);  // lanes [0, B) may be needed
        const uint32_t x = psx_mulhi32(word, err_N);
        const bool live = lane < B && t < TMAX;
        const uint32_t h = (x * 0x9E3779B1u) >> 21;
        const uint32_t seen = live ? atomicOr(&bits[h >> 5], 1u << (h & 31u)) & (1u << (h & 31u)) : 0u;
        unsigned long long dupm = 0;
        if constexpr (FLAGGED) {
            // lanes that found their bit set: of the lanes that name one index all but one did
            for (unsigned long long left = __ballot(seen != 0u); left;) {
                const uint32_t xq = (uint32_t)__builtin_amdgcn_readlane((int)x, __ffsll((long long)left) - 1);
                const unsigned long long same = __ballot(live && x == xq);
                left &= ~same;
                bool d = false;
                for (uint32_t q = lane; q < cnt; q += 64u) d |= (list[q] & 0xFFFFFu) == xq;
                dupm |= __ballot(d) ? same : same & (same - 1ull);
            }
        } else if (__ballot(seen != 0u)) {  // the batch's and the earlier batches'
            for (uint32_t q = 0; q + 1u < B; ++q) {
                const uint32_t xq = (uint32_t)__builtin_amdgcn_readlane((int)x, (int)q);
                dupm |= __ballot(live && x == xq) & (~0ull << (q + 1u));
            }
            bool d = false;
            for (uint32_t q = 0; q < cnt; ++q) d |= (list[q] & 0xFFFFFu) == x;
            dupm |= __ballot(live && d);
        }
        const bool fresh = live && !((dupm >> lane) & 1ull);
        const unsigned long long m = __ballot(fresh);
        const uint32_t rank =
            cnt + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
        if (fresh && rank < K) list[rank] = x | ((((word & 0xFFFFu) * 3u) >> 16) << 20);
        cnt = min(K, cnt + (uint32_t)__popcll(m));
        if (cnt == K) break;
        t0 += B;
        wave_sync();  // list entries of this batch seen by every lane
    }
    return cnt;
}

// Records of one position shared by several records, from index i (the
// oracle's seq_read step): the first carried SNV sets the true base, the
// read's error there (summary e; base index p + boff) substitutes it, every
// record gains depth and each SID head an alternative read when its
// alternative is observed (SNV) or carried (indel). Returns the index past
// the position.
template <class V>
__device__ __forceinline__ uint32_t count_group(const job_dev& J, const V& v, uint32_t i, uint32_t allele,
                                                uint32_t leaf, const terr& e, uint32_t boff) {
    const uint32_t p = v.pos[i];
    const uint32_t g0 = i;
    uint32_t g1 = i + 1;
    while (g1 < v.n && v.pos[g1] == p) ++g1;
    uint32_t tb = PSX_INFO_REF(v.info[g0]);
    for (uint32_t q = g0; q < g1; ++q) {
        const uint32_t in = v.info[q];
        if (PSX_INFO_KIND(in) == PSX_SNV && PSX_INFO_ALLELE(in) == allele && carried(J, in, v.lo[q], v.hi[q], leaf)) {
            tb = PSX_INFO_ALT(in);
            break;
        }
    }
    const uint32_t ob = observe(e, p + boff, tb);
    for (uint32_t q = g0; q < g1; ++q) {
        v.add_dep(q);
        const uint32_t in = v.info[q];
        if (!PSX_INFO_HEAD(in)) continue;
        if (PSX_INFO_KIND(in) == PSX_SNV) {
            if (ob == PSX_INFO_ALT(in)) v.add_alt(q);
        } else {
            bool car = false;
            for (uint32_t q2 = q; q2 < g1 && (q2 == q || !PSX_INFO_HEAD(v.info[q2])); ++q2) {
                const uint32_t in2 = v.info[q2];
                car |= PSX_INFO_ALLELE(in2) == allele && carried(J, in2, v.lo[q2], v.hi[q2], leaf);
            }
            if (car) v.add_alt(q);
        }
    }
    return g1;
}

// A sequencing error of a slow template replacing the true base at the
// position of record i (the first of its position) by substitution index
// sub: the counts took the true base there, so each SNV head changes its
// alternative count by [observed == alt] - [true == alt]. Depth and indel
// counts do not depend on the observed base.
template <class V>
__device__ __forceinline__ void error_fix(const job_dev& J, const V& v, uint32_t i, uint32_t allele, uint32_t leaf,
                                          uint32_t sub) {
    const uint32_t p = v.pos[i];
    uint32_t g1 = i + 1;
    while (g1 < v.n && v.pos[g1] == p) ++g1;
    uint32_t tb = PSX_INFO_REF(v.info[i]);
    for (uint32_t q = i; q < g1; ++q) {
        const uint32_t in = v.info[q];
        if (PSX_INFO_KIND(in) == PSX_SNV && PSX_INFO_ALLELE(in) == allele && carried(J, in, v.lo[q], v.hi[q], leaf)) {
            tb = PSX_INFO_ALT(in);
            break;
        }
    }
    const uint32_t ob = sub < tb ? sub : sub + 1u;
    for (uint32_t q = i; q < g1; ++q) {
        const uint32_t in = v.info[q];
        if (!PSX_INFO_HEAD(in) || PSX_INFO_KIND(in) != PSX_SNV) continue;
        const int d = (ob == PSX_INFO_ALT(in) ? 1 : 0) - (tb == PSX_INFO_ALT(in) ? 1 : 0);
        if (d) v.add_alt_n(q, d);
    }
}

// Stratum geometry shared by both kernels.
struct stratum {
    uint32_t b, e, wend, k0, n_win;
    uint64_t nj, before;
};

// Records of the stratum index from stratum j's first to the last that a read
// below wend can reach (up to the end of wend's stratum).
__device__ __forceinline__ uint32_t window_records(const job_dev& J, const seg_dev& S, uint32_t k0, uint32_t wend) {
    const uint32_t last = (S.len + PSX_STRATUM - 1) / PSX_STRATUM;
    return uniform_at(J.bucket, S.bucket_off + min((wend + PSX_STRATUM - 1) / PSX_STRATUM, last)) - k0;
}

__device__ __forceinline__ stratum stratum_of(const job_dev& J, const seg_dev& S, uint32_t j) {
    stratum s;
    s.b = j * PSX_STRATUM;
    s.e = min(s.b + PSX_STRATUM, S.W);
    s.before = templates_below(S, s.b);
    s.nj = templates_below(S, s.e) - s.before;
    s.wend = min(S.len, s.e - 1 + J.reach);
    s.k0 = uniform_at(J.bucket, S.bucket_off + j);
    s.n_win = window_records(J, S, s.k0, s.wend);
    return s;
}

// The segment's first entry of the count arrays.
__device__ __forceinline__ uint64_t out_off(const job_dev& J, const seg_dev& S) { return (uint64_t)S.so * J.n_mut; }

// The read kernel's window: only the SNVs of [k0, k0 + n_win) that a read of
// the segment's output sample can carry (present flags), compacted in table
// order, with the bucket index over them; returns their number. Reads take
// their bases from the first carried SNV at each position, so the records
// left out (indels, records no source of the sample carries) never change a
// read. s_cnt: one word per wave.
template <int BLOCK, int CAP>
__device__ __forceinline__ uint32_t stage_snvs(const job_dev& J, const seg_dev& S, const stratum& s, uint32_t* s_pos,
                                               uint32_t* s_lo, uint32_t* s_hi, uint32_t* s_info, uint16_t* s_bucket,
                                               uint32_t* s_cnt, uint32_t tid) {
    constexpr uint32_t WAVES = BLOCK / 64;
    const uint8_t* pres = J.present + (uint64_t)S.so * J.n_mut + s.k0;
    const uint32_t wave = tid >> 6;
    uint32_t n = 0;  // block-uniform
    for (uint32_t c = 0; c < s.n_win; c += BLOCK) {
        const uint32_t i = c + tid;
        const bool in = i < s.n_win;
        const uint32_t info = in ? J.info[s.k0 + i] : 0u;
        const uint32_t pos = in ? J.pos[s.k0 + i] : 0u, lo = in ? J.lo[s.k0 + i] : 0u, hi = in ? J.hi[s.k0 + i] : 0u;
        const bool keep = in && PSX_INFO_KIND(info) == PSX_SNV && pres[i] != 0;
        const unsigned long long m = __ballot(keep);
        if ((tid & 63u) == 0) s_cnt[wave] = (uint32_t)__popcll(m);
        __syncthreads();
        uint32_t off = n, tot = 0;
#pragma unroll
        for (uint32_t w = 0; w < WAVES; ++w) {
            const uint32_t cw = s_cnt[w];
            off += w < wave ? cw : 0u;
            tot += cw;
        }
        if (keep) {
            const uint32_t r =
                off + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
            s_pos[r] = pos;
            s_lo[r] = lo;
            s_hi[r] = hi;
            s_info[r] = info;
        }
        n += tot;
        __syncthreads();
    }
    const uint32_t nb = ((s.wend - s.b) >> NB_SHIFT) + 1;
    for (uint32_t q = tid; q < nb; q += BLOCK) {
        const uint32_t target = s.b + (q << NB_SHIFT);
        uint32_t a = 0, z = n;
        while (a < z) {
            const uint32_t mid = (a + z) >> 1;
            if (s_pos[mid] < target) a = mid + 1; else z = mid;
        }
        s_bucket[q] = (uint16_t)a;
    }
    __syncthreads();
    return n;
}

// Presence (the sample holds the mutation) and zeroed counters; also resets
// the work counter of the count kernel that follows on the stream.
// Whether record m can be carried by a read of output sample P: a leaf of the
// sample lies in its leaf range, or the normal genome carries it and the
// sample's reads can come from the normal genome (the normal sample, or purity
// below 1). Oracle: the presence flags of orc_simulate_seq.
__device__ __forceinline__ bool record_present(const job_dev& J, const pres_dev& P, uint64_t m) {
    const uint32_t info = J.info[m];
    const uint32_t nat = PSX_INFO_NATURE(info);
    const bool normal_has = nat == PSX_GERMINAL || (nat == PSX_PRENEOPLASTIC && J.preneo);
    bool pres;
    if (P.n_cells == 0) {
        pres = normal_has;
    } else {
        pres = J.purity_lt1 && normal_has;
        if (!pres) {
            pres = cells_below(J, P.sample, J.hi[m]) > cells_below(J, P.sample, J.lo[m]);
        }
    }
    return pres;
}

// The (output sample, mutation) pair of thread q: ps lists each pair range's
// first index.
__device__ __forceinline__ const pres_dev& pres_of(const pres_dev* __restrict__ ps, uint32_t n_ps, uint64_t q) {
    uint32_t a = 0, z = n_ps;
    while (a < z) {
        const uint32_t mid = (a + z) >> 1;
        if (ps[mid].begin <= q) a = mid + 1; else z = mid;
    }
    return ps[a - 1];
}

__global__ void __launch_bounds__(256) k_seq_init(const job_dev* __restrict__ jobs, const pres_dev* __restrict__ ps,
                                                  uint32_t n_ps, uint64_t total,
                                                  unsigned long long* __restrict__ queue, uint32_t n_jobs) {
    const uint64_t q = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q == 0) {
        queue[0] = 0ull;  // the sparse jobs' item counter
        queue[1] = 0ull;  // the others'
        for (uint32_t k = 0; k < n_jobs; ++k)
            if (jobs[k].acc) *jobs[k].acc = 0ull;
    }
    if (q >= total) return;
    const pres_dev P = pres_of(ps, n_ps, q);
    const job_dev& J = jobs[P.job];
    const uint64_t m = q - P.begin;
    const uint64_t o = (uint64_t)P.so * J.n_mut + m;
    J.alt[o] = 0;
    J.depth[o] = 0;
    J.present[o] = record_present(J, P, m) ? 1 : 0;
}

// Presence flags only (read materialisation: the read kernel stages the SNVs
// a read of the sample can carry).
__global__ void __launch_bounds__(256) k_reads_present(const job_dev* __restrict__ jobs,
                                                       const pres_dev* __restrict__ ps, uint32_t n_ps, uint64_t total) {
    const uint64_t q = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= total) return;
    const pres_dev P = pres_of(ps, n_ps, q);
    const job_dev& J = jobs[P.job];
    const uint64_t m = q - P.begin;
    J.present[(uint64_t)P.so * J.n_mut + m] = record_present(J, P, m) ? 1 : 0;
}

// --------------------------------------------------- read materialisation
//
// Work layout. A wave takes 64 templates of the stratum at a time (one per
// lane: draws, insert, source leaf), then writes their reads in passes of 64
// reads, one read per lane, in output order: with paired ends lane l of pass
// p holds mate l % 2 of template p * 32 + l / 2, whose fields it fetches from
// the lane that drew it. A read is built in the lane's row of a wave-private
// LDS stage and each pass is copied out by the whole wave with 16-byte
// coalesced stores, so no block barrier separates generation from the copy.

// One read into row[0 .. 2 + ceil(L/16)): word 0 = start, word 1 = leaf |
// allele << 26 | mate << 30 | (errors > 0) << 31, then the 2-bit bases (base
// i of the read in bits 2 (i % 16) of word 2 + i / 16) taken from the staged
// reference (s_ref[0] is reference word ref_b / 16), with the first carried
// SNV at each position and the template summary's errors of this mate
// applied; bases past the read end are 0. A slow template's errors are
// applied to the row afterwards (apply_error). Oracle: read_row.
template <int NW, class V>
__device__ __forceinline__ void write_read(const job_dev& J, const V& v, uint32_t x, uint32_t leaf, uint32_t allele,
                                           uint32_t mate, const terr& e, const uint32_t* s_ref, uint32_t ref_b,
                                           uint32_t* row) {
    const uint32_t tail = J.L & 15u;
    const uint32_t xr = x - ref_b;
    const uint32_t w = xr >> 4;
    const uint32_t sh = (xr & 15u) * 2u;
    // s_ref holds one word past the staged range, so w + k + 1 is always readable
    if constexpr (NW > 0) {
        // 16-byte row: bases built in registers, stored as three 128-bit writes
        uint32_t wd[NW];
#pragma unroll
        for (int k = 0; k < NW; ++k) wd[k] = __builtin_amdgcn_alignbit(s_ref[w + k + 1], s_ref[w + k], sh);
        if (tail) wd[NW - 1] &= (1u << (2u * tail)) - 1u;
        static_assert((NW + 2) % 4 == 0, "rows of whole 16-byte vectors");
        uint4* r4 = reinterpret_cast<uint4*>(row);
        r4[0] = uint4{x, 0u, wd[0], wd[1]};
#pragma unroll
        for (int q = 1; q < (NW + 2) / 4; ++q) r4[q] = uint4{wd[4 * q - 2], wd[4 * q - 1], wd[4 * q], wd[4 * q + 1]};
    } else {
        const uint32_t nw = (J.L + 15u) >> 4;
        uint32_t lo = s_ref[w];
        for (uint32_t k = 0; k < nw; ++k) {
            const uint32_t hi = s_ref[w + k + 1];
            uint32_t word = __builtin_amdgcn_alignbit(hi, lo, sh);  // bits [sh, sh + 32) of hi:lo
            if (k + 1 == nw && tail) word &= (1u << (2u * tail)) - 1u;
            row[2 + k] = word;
            lo = hi;
        }
    }
    // SNVs at [x, x + L) in table order; the first carried SNV at a position
    // sets its base. One loop from the lane's bucket start (records before x
    // are passed over), uniform trip count, branch-free read-modify-writes of
    // the lane's own row (an unchanged word when nothing applies).
    const uint32_t end = x + J.L;
    uint32_t i = v.start(x);
    uint32_t p = v.n ? v.pos[v.at(i)] : end;  // at() needs n > 0
    bool go = i < v.n && p < end;
    uint32_t last = 0xFFFFFFFFu;
    while (__ballot(go)) {
        const uint32_t ic = go ? i : 0u;
        const uint32_t in = v.info[ic], lo = v.lo[ic], hi = v.hi[ic];
        i += go ? 1u : 0u;
        const uint32_t pn = v.pos[v.at(i)];
        const bool apply = go && p >= x && p != last && PSX_INFO_KIND(in) == PSX_SNV &&
                           PSX_INFO_ALLELE(in) == allele && carried(J, in, lo, hi, leaf);
        if (apply) {  // rare: only applying lanes touch their row (no bank conflicts from the others)
            const uint32_t o = p - x, s2 = (o & 15u) * 2u;
            row[2 + (o >> 4)] = (row[2 + (o >> 4)] & ~(3u << s2)) | (PSX_INFO_ALT(in) << s2);
        }
        last = apply ? p : last;
        go = go && i < v.n && pn < end;
        p = pn;
    }
    // the summary's errors on this mate (wave-uniform trip count, predicated)
    const uint32_t ne = e.n();
    uint32_t flag = 0;
    for (uint32_t q = 0; __ballot(q < ne); ++q) {
        const uint32_t eq = q == 0u ? (e.w01 & 0xFFFFu) : (q == 1u ? e.w01 >> 16 : e.w2n & 0xFFFFu);
        const uint32_t b = eq & 0x1FFFu;
        const uint32_t m = b >= J.L ? 1u : 0u;
        if (q < ne && m == mate) {
            const uint32_t o = b - m * J.L, s2 = (o & 15u) * 2u;
            const uint32_t wv = row[2 + (o >> 4)];
            const uint32_t tb = (wv >> s2) & 3u, sub = eq >> 13;
            const uint32_t nb = sub < tb ? sub : sub + 1u;
            row[2 + (o >> 4)] = (wv & ~(3u << s2)) | (nb << s2);
            flag = 1u;
        }
    }
    if constexpr (NW == 0) row[0] = x;
    row[1] = leaf | (allele << 26) | (mate << 30) | (flag << 31);
}

// A sequencing error at offset o of a written read: the base there is
// replaced by substitution index sub among the three other bases, and the
// read is flagged. ATOMIC: the row is shared with other lanes that may patch
// other bases of the same word at the same time (no two errors share a base,
// so the base read here is stable).
template <bool ATOMIC>
__device__ __forceinline__ void apply_error(uint32_t* row, uint32_t o, uint32_t sub) {
    uint32_t* wp = row + 2 + (o >> 4);
    const uint32_t s2 = (o & 15u) * 2u;
    const uint32_t tb = (*wp >> s2) & 3u;
    const uint32_t nb = sub < tb ? sub : sub + 1u;
    if (ATOMIC) {
        atomicXor(wp, (tb ^ nb) << s2);
        atomicOr(row + 1, 0x80000000u);
    } else {
        *wp ^= (tb ^ nb) << s2;
        row[1] |= 0x80000000u;
    }
}

// STAGE: reads are built in LDS and copied out per pass (read_words small
// enough for 64 rows per wave); otherwise each lane builds its read in place
// in the output. NW > 0: reads of NW base words (rows of whole 16-byte
// vectors, built in registers); NW = 0: any read size. CNA: segments with
// copy-number events keep only the templates whose copy slot is a copy of
// their source (their reads from J.cn_row on); the others as without. The
// 512-thread forms are held to 80 VGPRs (the copy-number one spills two), so
// that 3 blocks run per CU instead of 2: 5e7 single-end 100 bp reads 737 ->
// 615 us. Reads with copy numbers (2.7e7 of 3.3e7 templates' draws): a lane
// per draw, the kept ones packed between two barriers, 1,100 us; a lane per
// kept template, numbered by the bits of the pass that counts them, 450 us.
template <int BLOCK, int CAP, bool STAGE, int NW, bool CNA = false>
__global__ void __launch_bounds__(BLOCK, BLOCK == 512 ? 6 : 1) k_seq_reads(const seq_launch L) {
    constexpr uint32_t WAVES = BLOCK / 64;
    __shared__ uint32_t s_pos[CAP], s_lo[CAP], s_hi[CAP], s_info[CAP];
    __shared__ uint16_t s_bucket[NB_MAX];
    __shared__ uint32_t s_ref[REF_MAX];
    __shared__ lds_tables s_tab;
    __shared__ uint32_t s_run;
    __shared__ uint32_t s_cnt[WAVES];
    __shared__ uint32_t s_elist[WAVES][ELIST];  // per wave: errors of a slow template
    __shared__ cn_window s_cn;                  // CNA: the stratum's events; the chunk's kept templates per group and
    __shared__ uint64_t s_mask[CNA ? CN_CHUNK : 1u];      // those of the groups before
    __shared__ uint32_t s_below[CNA ? CN_CHUNK + 1u : 1u];
    extern __shared__ uint4 s_stage4[];  // STAGE: per wave 64 rows of read_words words
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63u, wave = tid >> 6;
    uint32_t* list = s_elist[wave];
    const uint32_t RW = L.read_words;
    const bool vec4 = L.out_vec4 != 0;  // RW % 4 == 0 and a 16-byte aligned output
    uint32_t* stage = reinterpret_cast<uint32_t*>(s_stage4) + wave * 64u * RW;
    const uint4* stage4 = reinterpret_cast<const uint4*>(stage);
    uint32_t in_tab = UNRESOLVED;  // the job whose tables s_tab holds
    for (uint32_t run = blockIdx.x;;) {
      const item_run R = run_of(L, run);
      if (R.first == R.end) break;
      if (tid == 0) s_run = gridDim.x + (uint32_t)atomicAdd(L.queue, 1ull);  // the block's next run
      for (uint32_t item = R.first; item < R.end; ++item) {
        const item_dev it = uniform_at(L.items, item);
        const seg_dev S = uniform_at(L.segs, it.seg);
        const job_dev J = uniform_at(L.jobs, S.job);
        const uint32_t c2 = (S.chr << 16) | S.so;
        const uint32_t rpt = J.pe ? 2u : 1u;
        const uint32_t tpp = 64u / rpt;  // templates per pass
        const uint32_t chr_words = (S.len + 15u) >> 4;
        if (in_tab != S.job) {
            in_tab = S.job;
            load_tables(J, s_tab, tid, BLOCK);
            __syncthreads();
        }
        for (uint32_t j = it.j0; j < it.j1; ++j) {
            const stratum s = stratum_of(J, S, j);
            const bool fits = s.n_win <= (uint32_t)CAP;
            // reference words covering [b, wend) plus one
            const uint32_t ref_w0 = s.b >> 4;
            const uint32_t n_ref = min(chr_words, ((s.wend + 15u) >> 4) + 1u) - ref_w0;
            for (uint32_t i = tid; i <= n_ref; i += BLOCK) s_ref[i] = i < n_ref ? J.packed[S.chr_woff + ref_w0 + i] : 0u;
            if (CNA && S.n_cna && wave == 0) cn_fill(J, S, s.b, s.e, lane, s_cn);
            uint32_t n_snv = 0;
            if (fits) n_snv = stage_snvs<BLOCK, CAP>(J, S, s, s_pos, s_lo, s_hi, s_info, s_bucket, s_cnt, tid);
            else __syncthreads();
            const lds_view lv{s_pos, s_lo, s_hi, s_info, s_bucket, n_snv, s.b};
            const glb_view gv{J.pos + s.k0, J.lo + s.k0, J.hi + s.k0, J.info + s.k0, nullptr, nullptr, s.n_win};
            const uint32_t nj = (uint32_t)s.nj;
            // Rounds of WAVES x 64 templates, 64 per wave: lanes [0, n_t) hold the templates (start tx, mate start tx2,
            // leaf | allele << 26, template index tr) whose reads start at read index first0. With copy-number events
            // only the templates whose copy slot is a copy of their source have reads: k_cn_accept left a bit for each;
            // they are numbered by chunks of CN_CHUNK groups of 64, and a lane finds its template by its number.
            const bool cn = CNA && S.n_cna != 0u;
            // the item's part of the stratum's templates (one part with copy numbers): [p0, p0 + part_n)
            uint32_t p0 = 0, part_n = nj;
            if (seg_parts(S) != 1u) {
                const uint32_t share = ((nj + seg_parts(S) - 1u) / seg_parts(S) + 63u) & ~63u;
                p0 = min(nj, it.part * share);
                part_n = min(share, nj - p0);
            }
            uint64_t row = cn ? uniform_at(J.cn_row, S.st_off + j) : S.read_base + (s.before + p0) * rpt;
            const uint32_t n_grp = cn ? (nj + 63u) >> 6 : 1u;
            for (uint32_t g0 = 0; g0 < n_grp; g0 += CN_CHUNK) {
            uint32_t nk = part_n;  // templates with reads (of the chunk)
            if (CNA && cn) {
                __syncthreads();  // the chunk before is done
                const uint64_t* const mask = L.cn_kept + S.read_base + (uint64_t)j * cn_groups(S) + g0;
                uint64_t m = 0;
                uint32_t n = 0;
                if (tid < CN_CHUNK) {
                    m = g0 + tid < n_grp ? mask[tid] : 0u;
                    s_mask[tid] = m;
                    n = (uint32_t)__popcll(m);
                    for (uint32_t k = 1; k < 64u; k <<= 1) {
                        const uint32_t v = (uint32_t)__shfl_up((int)n, k);
                        n += lane >= k ? v : 0u;
                    }
                    if (lane == 63u) s_cnt[wave] = n;
                }
                __syncthreads();
                if (tid < CN_CHUNK) {
                    for (uint32_t k = 0; k < wave; ++k) n += s_cnt[k];
                    s_below[tid + 1u] = n;
                    if (tid == 0) s_below[0] = 0;
                }
                __syncthreads();
                nk = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_below[CN_CHUNK]);
            }
            // The chunks of 64 templates are shifted by o so that every pass after the first chunk starts on a
            // 1024-byte boundary of the output (else 512, 256, 128): the first chunk holds the templates before the
            // first aligned row. A 16-byte offset of such 3 KiB passes costs about 10 % of the write rate (partly
            // written lines at every pass boundary).
            uint32_t o = 0;
            if (STAGE && vec4) {
                const uint64_t a0 = (uint64_t)(uintptr_t)(L.reads_out + row * RW);
                const uint64_t step = (uint64_t)rpt * RW * 4u;  // bytes per template
                for (uint32_t A = 1024u; A >= 128u; A >>= 1) {
                    const unsigned long long m = __ballot(((a0 + lane * step) & (A - 1u)) == 0u);
                    if (m) {
                        o = (64u - ((uint32_t)__ffsll((long long)m) - 1u)) & 63u;
                        break;
                    }
                }
            }
            for (uint32_t base = 0; base < nk + o; base += WAVES * 64u) {
                // the wave's chunk: templates [c0, cend) (virtual templates [vb, vb + 64) less o)
                const uint32_t vb = base + wave * 64u;
                const uint32_t c0 = vb == 0u ? 0u : vb - o;
                const uint32_t cend = min(vb + 64u - o, nk);
                const uint32_t n_t = cend > c0 ? cend - c0 : 0u;
                const uint64_t first0 = row + (uint64_t)c0 * rpt;
                uint32_t tx = 0, tx2 = 0, tla = 0, tr = p0 + c0 + lane;
                if (CNA && cn) {
                    if (lane < n_t) {
                        uint32_t a = 0;  // the group of kept template tr
                        for (uint32_t h = CN_CHUNK / 2u; h; h >>= 1) a += s_below[a + h] <= tr ? h : 0u;
                        tr = ((g0 + a) << 6) + nth_set(s_mask[a], tr - s_below[a]);
                        psx_u4 w;
                        tmpl t;
                        cn_template(J, S, s_cn, (uint32_t)__builtin_amdgcn_readfirstlane((int)s_cn.n), tr, j, s.b, s.e, w, t);
                        tx = t.x;
                        tx2 = mate_start(J, S, s_tab, t.x, w.w);
                        tla = (t.cell == S.n_cells ? J.n_leaves : J.sample_leaves[S.leaf_off + t.cell]) | (t.allele << 26);
                    }
                } else if (lane < n_t) {
                    tmpl t = make_template(J, S, s_tab, tr, j, s.b, s.e);
                    tx = t.x;
                    tx2 = t.x2;
                    tla = leaf_of(J, S, t) | (t.allele << 26);
                }
                if (n_t == 0) continue;
                const bool valid = lane < n_t;
                const uint32_t tr0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)tr);  // lane 0 holds a template
                const terr te = J.err_n ? template_errors(J, J.seed, s_tab.err, valid ? tr : tr0, j, c2, valid) : terr{0u, 0u};
                for (uint32_t p = 0; p < rpt; ++p) {
                    const uint32_t src = p * tpp + lane / rpt;
                    const uint32_t mate = lane & (rpt - 1u);
                    const uint32_t x1 = (uint32_t)__shfl((int)tx, (int)src);
                    const uint32_t x2 = (uint32_t)__shfl((int)tx2, (int)src);
                    const uint32_t la = (uint32_t)__shfl((int)tla, (int)src);
                    const terr e = shfl_terr(te, src);
                    const uint32_t t0 = p * tpp;  // first template of the pass
                    const uint32_t nt = t0 < n_t ? min(tpp, n_t - t0) : 0u;
                    const uint64_t first = first0 + (uint64_t)t0 * rpt;
                    uint32_t* row = STAGE ? stage + lane * RW : L.reads_out + (first + lane) * RW;
                    if (src < n_t) {
                        const uint32_t x = mate ? x2 : x1;
                        if (fits)
                            write_read<NW>(J, lv, x, la & 0x3FFFFFFu, la >> 26, mate, e, s_ref, ref_w0 << 4, row);
                        else
                            write_read<NW>(J, gv, x, la & 0x3FFFFFFu, la >> 26, mate, e, s_ref, ref_w0 << 4, row);
                    }
                    // slow templates of the pass (template lanes [t0, t0 + nt)): the wave generates each
                    // one's errors and patches its reads
                    unsigned long long sm = __ballot(te.slow() && lane >= t0 && lane < t0 + nt);
                    while (sm) {  // wave-uniform, rare
                        const uint32_t sl = (uint32_t)__ffsll((long long)sm) - 1u;
                        sm &= sm - 1ull;
                        // the slow template's index (contiguous without copy-number events)
                        const uint32_t rs = cn ? (uint32_t)__builtin_amdgcn_readlane((int)tr, (int)sl) : tr0 + sl;
                        wave_sync();
                        const uint32_t n_err = wave_template_errors(J.seed, J.err_n, J.err_k0, J.err_N, s_tab.err,
                                                                    rs, j, c2, list, lane);
                        wave_sync();  // list entries and (STAGE) every row of the pass written
                        for (uint32_t k0 = 0; k0 < n_err; k0 += 64u) {
                            const uint32_t k = k0 + lane;
                            const uint32_t w = k < n_err ? list[k] : 0u;
                            const uint32_t b = w & 0xFFFFFu, sub = w >> 20;
                            const uint32_t m = b >= J.L ? 1u : 0u;
                            const uint32_t o = b - m * J.L;
                            const uint32_t rl = (sl - t0) * rpt + m;  // the read's lane in the pass
                            const bool on = k < n_err;
                            if (STAGE) {
                                if (on) apply_error<true>(stage + rl * RW, o, sub);
                            } else {
                                // rows live in global memory: each lane patches its own read
                                for (uint32_t q = 0; q < 64u && k0 + q < n_err; ++q) {
                                    const uint32_t rq = (uint32_t)__shfl((int)rl, (int)q);
                                    const uint32_t oq = (uint32_t)__shfl((int)o, (int)q);
                                    const uint32_t sq = (uint32_t)__shfl((int)sub, (int)q);
                                    if (rq == lane) apply_error<false>(row, oq, sq);
                                }
                            }
                        }
                    }
                    if (STAGE) {
                        wave_sync();
                        const uint32_t words = nt * rpt * RW;
                        uint32_t* dst = L.reads_out + first * RW;
                        if (vec4) {
                            // plain stores: non-temporal ones cap this write pattern near 4.5 TB/s
                            uint4* d4 = reinterpret_cast<uint4*>(dst);
                            for (uint32_t q = lane; q < (words >> 2); q += 64u) d4[q] = stage4[q];
                        } else {
                            for (uint32_t q = lane; q < words; q += 64u) dst[q] = stage[q];
                        }
                        wave_sync();
                    }
                }
            }
            row += (uint64_t)nk * rpt;
            }
            __syncthreads();
        }
      }
      __syncthreads();
      run = __builtin_amdgcn_readfirstlane(s_run);
      __syncthreads();  // read by every wave before it is written again
    }
}

// Kept templates of every stratum of the segments with copy-number events
// (the read kernel's draws, so its row order follows), and a bit for each
// template: one wave per stratum, 64 templates at a time. Bound by vector
// instruction issue, 43 of them the draw's: a template's copies by a walk of
// the chromosome's events with its leaf's rank 261 us for 3.3e7 draws, by the
// stratum's events with ranges of cells 154 us.
struct accept_args {
    const job_dev* jobs;
    const seg_dev* segs;
    const uint32_t* cn_seg;    // segment index of each segment with events
    const uint32_t* cn_first;  // its first stratum (index into kept), n_seg + 1 entries
    uint32_t n_seg;
    uint64_t* kept;            // per stratum
    uint64_t* mask;            // with cn_mask: which templates are kept, 64 a word, cn_groups words a stratum
    const uint64_t* cn_mask;   // the first word of each segment with events (null: no masks)
};

__global__ void __launch_bounds__(256) k_cn_accept(const accept_args a) {
    const uint32_t g = (uint32_t)__builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4u + (threadIdx.x >> 6)));
    const uint32_t lane = threadIdx.x & 63u;
    if (g >= uniform_at(a.cn_first, a.n_seg)) return;  // the whole wave
    uint32_t lo = 0, hi = a.n_seg;  // the segment: the last k with cn_first[k] <= g
    while (hi - lo > 1u) {
        const uint32_t mid = (lo + hi) >> 1;
        if (uniform_at(a.cn_first, mid) <= g) lo = mid; else hi = mid;
    }
    const seg_dev S = uniform_at(a.segs, uniform_at(a.cn_seg, lo));
    const job_dev J = uniform_at(a.jobs, S.job);
    const uint32_t j = g - uniform_at(a.cn_first, lo);
    const uint32_t b = j * PSX_STRATUM, e = min(b + PSX_STRATUM, S.W);
    const uint64_t nj = templates_below(S, e) - templates_below(S, b);
    __shared__ cn_window s_cn[4];
    cn_window& cw = s_cn[threadIdx.x >> 6];
    cn_fill(J, S, b, e, lane, cw);
    wave_sync();
    const uint32_t n_ev = (uint32_t)__builtin_amdgcn_readfirstlane((int)cw.n);
    uint64_t* const mask = a.cn_mask ? a.mask + uniform_at(a.cn_mask, lo) + (uint64_t)j * cn_groups(S) : nullptr;
    uint64_t cnt = 0, mine = 0;  // 64 groups' masks, one per lane, stored together
    for (uint32_t q = 0; (uint64_t)q * 64u < nj; ++q) {
        const uint32_t r = q * 64u + lane;
        psx_u4 w;
        tmpl t;
        const bool ok = cn_template(J, S, cw, n_ev, r, j, b, e, w, t) && r < nj;
        const uint64_t m = __ballot(ok);
        cnt += (uint64_t)__popcll(m);
        mine = lane == (q & 63u) ? m : mine;
        if (mask && ((q & 63u) == 63u || (uint64_t)(q + 1u) * 64u >= nj) && lane <= (q & 63u)) mask[(q & ~63u) + lane] = mine;
    }
    if (lane == 0) a.kept[g] = cnt;
}

}  // namespace psxk
