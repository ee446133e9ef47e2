"""The work that users of this library have it do, as measurable cases.

A case is a dict of plain values; ``kind`` says which calls one pass makes:

* ``place``: mutation placement on one forest, the table brought to the host
  (Mutations.place, Mutations.download);
* ``place_seq``: placement on one forest, then a first look at it: count-only
  sequencing of the new table into device arrays (Mutations.place,
  simulate_seq_device);
* ``cohort``: many small forests over one reference placed in one call and
  sequenced in one batched launch (Mutations.place_batch,
  simulate_seq_batch);
* ``count``: count-only sequencing of a placed table into device arrays
  (simulate_seq_device; with ``vaf`` the VAF column too, seq_vaf_f32);
* ``reads``: every read materialised in device memory (simulate_seq_reads);
* ``serve``: a burst of requests through the serving runtime, results in host
  arrays (Server.submit, Server.wait).

The other fields are the sizes and options of the synthetic inputs:
``cells`` grown, ``samples`` tissue samples of ``leaves`` cells each, a
reference of ``bases`` over ``chroms`` chromosomes, passenger rates ``snv``
and ``indel`` per base per division, ``cov`` coverage, read size ``L``,
``insert`` mean insert size (0: single-end), ``err`` sequencing error rate,
``purity``, ``cna`` copy-number drivers with a whole-genome doubling,
``full`` engine options (ID signatures, timed exposures, drivers, germline and
preneoplastic mutations), ``jobs`` forests or requests.

torch is imported before the library, which then runs on torch's HIP runtime,
so outputs in device memory are returned as torch tensors over the library's
own buffers.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from process_amd import _abi as A
from process_amd import core, workloads

_PLAIN = dict(samples=1, chroms=1, snv=1e-8, indel=1e-9, cov=0.0, L=150, insert=350, err=1e-3, purity=1.0, cna=False,
              full=False, vaf=False, jobs=1)


def _case(kind: str, **kw) -> dict:
    return dict(_PLAIN, kind=kind, **kw)


def listed() -> list:
    return [
        # a biopsy-sized forest placed with every engine option in use: the smallest call, latency-bound
        _case("place", name="place_biopsy", cells=5_000, leaves=2_500, bases=10_000_000, full=True),
        # a new tumour placed and sequenced once at simulate_seq's defaults (10x, single-end 150 bp, no errors)
        _case("place_seq", name="place_tumour", cells=1_000_000, samples=3, leaves=10_000, bases=300_000_000, chroms=22,
              cov=10.0, insert=0, err=0.0),
        # a cohort of patients of uneven size over one reference, placed and sequenced in batched calls
        _case("cohort", name="cohort", cells=20_000, leaves=10_000, bases=50_000_000, chroms=4, cov=60.0, jobs=16),
        # the plain configuration: one small sample and the normal sample at 80x
        _case("count", name="count_small", cells=5_000, leaves=2_500, bases=10_000_000, indel=0.0, cov=80.0),
        # a targeted panel: few bases, deep, odd single-end reads, an impure sample, a high error rate
        _case("count", name="count_panel", cells=20_000, leaves=3_000, bases=1_500_000, chroms=3, snv=1e-7, cov=2000.0,
              L=101, insert=0, err=5e-3, purity=0.7),
        # the plain-large configuration: three 1e4-cell samples and the normal at 200x over 300 Mb, and the VAF column
        _case("count", name="count_large", cells=1_000_000, samples=3, leaves=10_000, bases=300_000_000, chroms=22,
              cov=200.0, vaf=True),
        # whole genomes with few mutations at ordinary depth: reads rarely cover a mutation
        _case("count", name="count_sparse", cells=40_000, samples=2, leaves=1_500, bases=200_000_000, chroms=22,
              snv=2e-9, indel=2e-10, cov=30.0, L=100, insert=300, err=2e-3),
        # copy-number segments and a doubled clone at purity 0.6 and 500x
        _case("count", name="count_cna", cells=100_000, leaves=10_000, bases=100_000_000, chroms=10, cov=500.0,
              purity=0.6, cna=True),
        # paired-end 150 bp reads of an exome-to-genome-sized run in HBM
        _case("reads", name="reads_pe150", cells=100_000, leaves=10_000, bases=100_000_000, chroms=10, cov=60.0),
        # single-end 100 bp reads: rows of an odd number of words
        _case("reads", name="reads_se100", cells=20_000, leaves=3_000, bases=50_000_000, chroms=4, cov=50.0, L=100,
              insert=0, err=2e-3),
        # reads of a copy-number-altered sample
        _case("reads", name="reads_cna", cells=20_000, leaves=3_000, bases=50_000_000, chroms=4, cov=40.0, purity=0.8,
              cna=True),
        # a burst of 16 requests of mixed size over four resident forests
        _case("serve", name="serve_burst", cells=100_000, samples=2, leaves=5_000, bases=50_000_000, chroms=4,
              cov=120.0, jobs=16),
    ]


def _nodes(cells: float, samples: int, leaves: float) -> float:
    """Nodes of a sampled birth-death forest (within 20 % of the generator's)."""
    return leaves * samples * (2.0 + max(0.0, math.log2(cells / (leaves * samples))))


def _muts(case: dict, share: float = 1.0) -> float:
    """Expected mutations of a forest whose cells and leaves are `share` of the case's."""
    return _nodes(case["cells"] * share, case["samples"], case["leaves"] * share) * 2.0 * case["bases"] * (
        case["snv"] + case["indel"])


def _shares(case: dict) -> list:
    """Sizes of the forests of a cohort, or of a server's resident forests, over the largest."""
    n = case["jobs"] if case["kind"] == "cohort" else 4
    return [math.exp(-3.0 * k / n) for k in range(n)]


def _covs(case: dict) -> list:
    """Coverage of each job or request: up to e^2 apart, the deepest first on the smallest forests."""
    return [case["cov"] * math.exp(-2.0 * ((7 * k + 3) % case["jobs"]) / case["jobs"]) for k in range(case["jobs"])]


def draw(rng) -> dict:
    def log(lo, hi):
        return math.exp(rng.uniform(math.log(lo), math.log(hi)))

    kind = rng.choice(["place", "place_seq", "cohort", "count", "count", "count", "reads", "reads", "serve"])
    bases = int(log(200_000, 250_000_000)) | 1
    cells = int(log(1_000, 600_000))
    samples = rng.choice([1, 1, 2, 3])
    leaves = max(40, min(int(cells / (2.0 * samples) * log(0.05, 1.0)), 12_000))
    chroms = rng.choice([1, 2, 5, 10, 22])
    cna = rng.random() < 0.25 and kind in ("count", "reads")
    pe = rng.random() < 0.6
    L = rng.choice([75, 100, 101, 125, 150, 151, 250])
    err = 0.0 if rng.random() < 0.2 else float("%.3g" % log(2e-4, 1e-2))
    purity = 1.0 if rng.random() < 0.5 else round(rng.uniform(0.3, 0.95), 2)
    # reads in all, then the coverage that gives them
    reads = log(1e5, {"place": 1e6, "place_seq": 5e7, "cohort": 3e8, "count": 8e8, "reads": 8e7, "serve": 3e8}[kind])
    jobs = rng.choice([3, 8, 13, 16]) if kind in ("cohort", "serve") else 1
    if kind in ("cohort", "serve"):
        bases, cells = min(bases, 60_000_001), min(cells, 50_000)
        leaves = min(leaves, max(40, cells // (2 * samples)))
        samples = 1 if kind == "cohort" else samples
    if kind == "place_seq":
        pe, err, purity = False, 0.0, 1.0
    # the table's size (from hundreds of records to a million, at most one per 100 bases), then the rate that gives it
    muts = min(log(300, 1e6), bases / 100.0)
    snv = float("%.3g" % (muts / (2.2 * _nodes(cells, samples, leaves) * bases)))
    cov = min(3000.0, reads * L / (float(bases) * jobs * (samples + 1)))
    return _case(kind, cells=cells, samples=samples, leaves=leaves, bases=bases, chroms=chroms, snv=snv,
                 indel=float("%.3g" % (snv / 10)), cov=round(max(cov, 0.1), 3), L=L, insert=(2 * L + 50) if pe else 0,
                 err=err, purity=purity, cna=cna, full=kind == "place" and rng.random() < 0.5,
                 vaf=kind == "count" and rng.random() < 0.5, jobs=jobs)


# ------------------------------------------------------------------- inputs

class _Over:
    """A library device buffer as torch.as_tensor takes it (no copy; the tensor keeps the buffer alive)."""

    def __init__(self, buf: core.DeviceArray):
        self.buf = buf
        kind = {1: "|u1", 4: "<f4" if buf.dtype.kind == "f" else "<i4"}[buf.dtype.itemsize]
        self.__cuda_array_interface__ = {"shape": buf.shape, "typestr": kind, "data": (buf.ptr, False), "version": 2}


def _tensor(buf: core.DeviceArray) -> torch.Tensor:
    return torch.as_tensor(_Over(buf), device="cuda")


class _Arrays:
    """The device arrays a session sequences into, [output sample][mutation], with room for any table of the case: the
    library fills the first samples x mutations entries. As a job it is one of a batched launch."""

    def __init__(self, ctx, case: dict, cap: int, genome=None, forest=None, seed: int = 0, **seq):
        self.cap, self.genome, self.forest, self.muts, self.seed, self.seq = cap, genome, forest, None, seed, seq
        shape = (case["samples"] + 1, cap)
        self.alt = core.DeviceArray(ctx, shape, np.int32).fill(0)
        self.depth = core.DeviceArray(ctx, shape, np.int32).fill(0)
        self.present = core.DeviceArray(ctx, shape, np.uint8).fill(0)
        self.out = [_tensor(self.alt), _tensor(self.depth), _tensor(self.present)]

    def take(self, table: core.Mutations) -> core.Mutations:
        if table.n > self.cap:
            raise ValueError(f"{table.n} mutations, room for {self.cap}")
        self.muts = table
        return table


def _room(muts: float) -> int:
    return int(1.3 * muts + 8.0 * math.sqrt(muts)) + 400


def _seq(case: dict, cov: float | None = None) -> dict:
    return dict(coverage=float(case["cov"] if cov is None else cov), read_size=case["L"], insert_size_mean=case["insert"],
                insert_size_stddev=10, error_rate=case["err"], purity=case["purity"], with_normal_sample=True)


def _forest(ctx, rng, cells: int, samples: int, leaves: int) -> core.Forest:
    """Two species (growth 0.2; driver 0.3 introduced early), samples of `leaves` cells."""
    fd = core.synth_forest(growth=[0.2, 0.3], death=[0.01, 0.01], intro_at=[0, max(2, min(1000, cells // 5))],
                           n_cells=cells, n_samples=samples, sample_size=leaves, seed=int(rng.integers(1 << 31)))
    return core.Forest(ctx, fd["cell_id"], fd["parent"], fd["species"], fd["sample"], fd["birth"], fd["n_samples"])


def _engine(case: dict, rng, genome: core.Genome) -> dict:
    # the context index at the engine's default sampling, or every site where the table needs them
    sampling = 100 if _muts(case) * 1000.0 < case["bases"] else 1
    eng = dict(snv_rate=[case["snv"]] * 2, indel_rate=[case["indel"]] * 2, sbs=rng.dirichlet(np.ones(96), size=1),
               epoch_start=[0.0], exposure=[[1.0]], n_pre_snv=0, n_pre_indel=0, pre_sbs=0, indel_max_len=10,
               indel_len_p=0.5, infinite_sites=True, ploidy=2, drivers=[], germline=[], context_sampling=sampling)
    lens = genome.lengths
    if case["full"]:
        packed: dict = {}
        pos = int(lens[0]) // 2
        c = len(lens) - 1
        germ = sorted({int(p) for p in rng.integers(0, int(lens[-1]), 50)} - {pos})
        eng.update(sbs=rng.dirichlet(np.ones(96), size=3), epoch_start=[0.0, 20.0],
                   exposure=rng.dirichlet(np.ones(3), size=2), n_pre_snv=40, n_pre_indel=10,
                   id_sig=rng.dirichlet(np.ones(A.PSX_ID_CLASSES), size=2),
                   id_exposure=rng.dirichlet(np.ones(2), size=2), pre_id=0,
                   drivers=[(1, 0, pos, (workloads.base_at(genome, packed, 0, pos) + 1) % 4, -1)],
                   germline=[(c, p, (workloads.base_at(genome, packed, c, p) + 2) % 4, k % 2) for k, p in enumerate(germ)])
    if case["cna"]:
        segs = np.random.default_rng(case["bases"])  # the tumour's karyotype goes with its reference
        eng["cna"] = (workloads.cna_segments(lens, segs, 8, 0) + [(1, 0, 0, 0, 0, A.PSX_CNA_WGD, 0)]
                      + workloads.cna_segments(lens, segs, 4, 1))
    return eng


def prepare(case: dict, seed: int) -> dict:
    """What a session holds before the call: the reference with its indexes (built by the engine's first placement),
    the forests, the tables already placed, the device arrays that receive the results."""
    ctx = core.default_context()
    rng = np.random.default_rng(seed)
    lens = workloads.log_uniform_lengths(case["chroms"], case["bases"], 1.0, 6.0, np.random.default_rng(case["chroms"]))
    genome = core.Genome(ctx, lens, seed=int(rng.integers(1 << 31)))
    eng = _engine(case, rng, genome)
    st = dict(case=case, ctx=ctx, genome=genome, engine=eng, seed=int(rng.integers(1 << 31)), seq=_seq(case))
    kind = case["kind"]
    if kind in ("cohort", "serve"):
        shares = _shares(case)
        forests = st["forests"] = [
            _forest(ctx, rng, max(100, int(case["cells"] * q) + 1), case["samples"], max(20, int(case["leaves"] * q)))
            for q in shares]
        seeds = st["place_seeds"] = [int(x) for x in rng.integers(1 << 31, size=len(shares))]
        seq_seeds = [int(x) for x in rng.integers(1 << 31, size=case["jobs"])]
        room = [_muts(case, q) for q in shares]
        if kind == "cohort":
            genome.context_index(eng["context_sampling"])
            st["jobs"] = [_Arrays(ctx, case, _room(m), genome, f, s, **_seq(case, c))
                          for m, f, s, c in zip(room, forests, seq_seeds, _covs(case))]
            return st
        # resident tables: exported records, a fixed number of each forest's, uploaded again
        st["tables"] = []
        placed = core.Mutations.place_batch(ctx, genome, forests, seeds, [eng] * len(shares))
        for f, m, want in zip(forests, placed, room):
            recs = m.download()
            keep = min(len(recs), max(1, int(0.7 * want - 4.0 * math.sqrt(want))))
            st["tables"].append(core.Mutations.upload(ctx, f, recs[np.sort(rng.permutation(len(recs))[:keep])]))
        st["requests"] = [(k % len(shares), s, _seq(case, c))
                          for k, s, c in zip(range(case["jobs"]), seq_seeds, _covs(case))]
        st["server"] = core.Server(ctx, 1 << 30)
        return st
    forest = st["forest"] = _forest(ctx, rng, case["cells"], case["samples"], case["leaves"])
    st["place_seed"] = int(rng.integers(1 << 31))
    cap = _room(_muts(case) + 110.0)
    if kind in ("place", "place_seq"):
        # the engine's first placement builds the reference's indexes
        core.Mutations.place(ctx, genome, forest, st["place_seed"] + 1, **eng).close()
        if kind == "place":
            st["recs"] = np.zeros((cap, 9), np.int32)
        else:
            st["arrays"] = _Arrays(ctx, case, cap)
        return st
    m = st["table"] = core.Mutations.place(ctx, genome, forest, st["place_seed"], **eng)
    if kind == "reads":
        n = core.num_reads(genome, forest, **st["seq"]) * (3 if case["cna"] else 1)
        st["buf"] = core.DeviceArray(ctx, (max(n, 1), core.read_words(**st["seq"])), np.uint32).fill(0)
        st["out"] = _tensor(st["buf"])
        return st
    st["arrays"] = _Arrays(ctx, case, cap)
    st["arrays"].take(m)
    if case["vaf"]:
        st["vaf"] = core.DeviceArray(ctx, st["arrays"].alt.shape, np.float32).fill(0)
        st["arrays"].out.append(_tensor(st["vaf"]))
    return st


def run(st: dict):
    """One pass through the library's calls."""
    case, ctx, genome = st["case"], st["ctx"], st["genome"]
    kind = case["kind"]
    if kind == "place":
        m = core.Mutations.place(ctx, genome, st["forest"], st["place_seed"], **st["engine"])
        st["recs"][:m.n] = m.download().view(np.int32).reshape(-1, 9)
        return st["recs"]
    if kind == "cohort":
        tables = core.Mutations.place_batch(ctx, genome, st["forests"], st["place_seeds"],
                                            [st["engine"]] * len(st["forests"]))
        for job, m in zip(st["jobs"], tables):
            job.take(m)
        n = core.simulate_seq_batch(ctx, st["jobs"])
        return [j.out for j in st["jobs"]] + [n]
    if kind == "reads":
        _, n = core.simulate_seq_reads(ctx, genome, st["forest"], st["table"], st["seed"], out=st["buf"], **st["seq"])
        return [st["out"], n]
    if kind == "serve":
        server = st["server"]
        tickets = [server.submit(genome, st["forests"][k], st["tables"][k], s, **seq) for k, s, seq in st["requests"]]
        got = [server.wait(t) for t in tickets]
        return [[a, d, p] for a, d, p, _ in got] + [np.array([s["n_reads"] for *_, s in got], np.int64)]
    arr = st["arrays"]
    m = st["table"] if kind == "count" else arr.take(
        core.Mutations.place(ctx, genome, st["forest"], st["place_seed"], **st["engine"]))
    n = core.simulate_seq_device(ctx, genome, st["forest"], m, st["seed"], arr.alt, arr.depth, arr.present, **st["seq"])
    if case["vaf"]:
        core.seq_vaf_f32(ctx, m, arr.alt, arr.depth, arr.present, out=st["vaf"])
    return arr.out + [n]


def exact(case: dict, seed: int):
    """No 64-bit restatement: every output is counted or drawn in integers, and the VAF column is one division of two of
    them, which can only be restated from the counts themselves."""
    return None


def work(case: dict) -> dict:
    """What a pass cannot do without. Placement: each forest node's 12 bytes read, each mutation's record (36 bytes) and
    the four words the sequencing kernels read written once. Sequencing: the 16 bytes of each record read and 9 per
    output sample written; one Philox4x32-10 draw per template (10 rounds of two 32x32->64 multiplies, two three-input
    xors and two key additions: 100 integer operations), one more for its errors. Materialised reads: each row written
    once. Sizes of the tables are expectations."""
    kind = case["kind"]
    out = case["samples"] + 1
    mates = 2 if case["insert"] else 1
    per_cov = case["bases"] * out / (case["L"] * mates)  # templates at coverage 1
    if kind in ("cohort", "serve"):
        sizes = _shares(case)
        nodes = sum(_nodes(case["cells"] * q, case["samples"], case["leaves"] * q) for q in sizes)
        muts = sum(_muts(case, q) for q in sizes)
        templates = sum(_covs(case)) * per_cov
    else:
        nodes, muts, templates = _nodes(case["cells"], case["samples"], case["leaves"]), _muts(case), case["cov"] * per_cov
    place = {"bytes": nodes * 12.0 + muts * 52.0, "flops": 100.0 * nodes + 200.0 * muts}
    draws = 100.0 * templates * (2.0 if case["err"] else 1.0)
    count = muts * (16.0 + 9.0 * out)
    if kind == "place":
        return {"bytes": place["bytes"] + muts * 36.0, "flops": place["flops"]}
    if kind in ("place_seq", "cohort"):
        return {"bytes": place["bytes"] + count, "flops": place["flops"] + draws}
    if kind == "count":
        return {"bytes": count, "flops": draws}
    if kind == "serve":
        return {"bytes": count * case["jobs"] / len(sizes), "flops": draws}
    row = 4.0 * (2 + (case["L"] + 15) // 16)
    return {"bytes": templates * mates * row + muts * 16.0 + case["bases"] / 4.0, "flops": draws}
