"""Launch shapes of the sequencing kernels against the oracle, bit for bit, at
the sizes where a launch rule changes."""
from __future__ import annotations

import numpy as np
import pytest

import cases
from oracle import oracle as O
from process_amd import core

pytestmark = pytest.mark.gpu


class World:
    """A two-species forest over a synthetic reference; the table is the GPU's own (its parity is tested elsewhere)."""

    def __init__(self, ctx, lens, forest_kw, snv, seed=5, **eng):
        self.lens = np.asarray(lens, np.uint32)
        self.g = core.Genome(ctx, self.lens, seed=seed)
        fd = cases.forest(**forest_kw)
        self.of = O.Forest(fd["cell_id"], fd["parent"], fd["species"], fd["sample"], fd["birth"], fd["n_samples"])
        self.pf = core.Forest(ctx, fd["cell_id"], fd["parent"], fd["species"], fd["sample"], fd["birth"],
                              fd["n_samples"])
        kw = dict(snv_rate=[snv, snv], indel_rate=[snv / 10, snv / 10], sbs=cases.signatures(1, 2), epoch_start=[0.0],
                  exposure=[[1.0]], n_pre_snv=8, n_pre_indel=4)
        kw.update(eng)
        self.pm = core.Mutations.place(ctx, self.g, self.pf, seed + 1, **kw)
        self.recs = self.pm.download()

    def check(self, got, seed, kw):
        oa, od, op, on = O.simulate_seq(self.lens, self.of, self.recs, seed, **kw)
        a, d, p = got
        assert np.array_equal(d, od) and np.array_equal(a, oa) and np.array_equal(p, op), kw
        return on


def test_runs_of_many_small_items(ctx):
    """A launch of many strata with few templates each is handed out in runs of several strata, which cross segments
    and jobs: 200 Mb over 22 chromosomes at 0.2-0.5x, three jobs of different read sizes, inserts and error rates."""
    lens = np.full(22, 200_000_000 // 22) + np.arange(22) * 1000
    w = World(ctx, lens, dict(n_cells=300, n_samples=2, sample_size=50, seed=3), 3e-9)
    spec = [dict(coverage=0.3, read_size=150, insert_size_mean=350, insert_size_stddev=10, error_rate=1e-2),
            dict(coverage=0.5, read_size=100, error_rate=2e-2, purity=0.6),
            dict(coverage=0.2, read_size=75, insert_size_mean=200, insert_size_stddev=5)]
    jobs = [core.SeqJob(ctx, w.g, w.pf, w.pm, 40 + k, **kw) for k, kw in enumerate(spec)]
    n = core.simulate_seq_batch(ctx, jobs)
    assert n == sum(w.check(j.results(), 40 + k, kw) for k, (j, kw) in enumerate(zip(jobs, spec)))
    # materialised reads: a chromosome's rows of the whole run are the oracle's reads of that chromosome alone
    kw = dict(spec[0], with_normal_sample=False, samples=[1])
    rows, n = core.simulate_seq_reads(ctx, w.g, w.pf, w.pm, 7, **kw)
    per = [core.num_reads(w.g, w.pf, **dict(kw, chromosomes=[c])) for c in range(22)]
    assert n == sum(per)
    first = sum(per[:21])
    alone = O.simulate_reads(w.lens, w.g.download(), w.of, w.recs, 7, per[21], **dict(kw, chromosomes=[21]))
    assert len(alone) == per[21] and np.array_equal(rows.numpy()[first:first + per[21]], alone)


@pytest.mark.parametrize("cov,kw", [
    # windows of one stratum in several rounds, of 2 and 4 strata, of 8 (no errors), single- and paired-end
    (900.0, dict(read_size=150, insert_size_mean=350, insert_size_stddev=10, error_rate=1e-3)),
    (45.0, dict(read_size=100, insert_size_mean=250, insert_size_stddev=15, error_rate=4e-3, purity=0.6)),
    (20.0, dict(read_size=151, error_rate=1e-3, purity=0.8, preneoplastic_in_normal=True)),
    (4.0, dict(read_size=75)),
    # nearly every template with repeated or more than three errors, more of them at records than a round lists
    (300.0, dict(read_size=120, insert_size_mean=300, insert_size_stddev=12, error_rate=0.05)),
    # mates far from their reads
    (60.0, dict(read_size=60, insert_size_mean=2500, insert_size_stddev=40, error_rate=1e-3, purity=0.0))])
def test_windows_of_dense_tables(ctx, dense, cov, kw):
    """Tables whose reads cover many positions are counted by windows (k_count_dense): strata per window, rounds, parts
    of an item, chromosomes of a few starts, records that share positions, the normal genome."""
    for w in dense:
        a, d, p, n = core.simulate_seq_arrays(ctx, w.g, w.pf, w.pm, 17, coverage=cov, **kw)
        assert n == w.check((a, d, p), 17, dict(kw, coverage=cov)) and d.sum() > 0


@pytest.fixture(scope="module")
def dense(ctx):
    forest = dict(n_cells=600, n_samples=2, sample_size=70, seed=6)
    lens = [70_001, 33_000, 8_192 + 149, 400, 153]
    return [World(ctx, lens, forest, 3e-5, n_pre_snv=60),
            World(ctx, [50_000, 2_600], forest, 4e-5, seed=8, infinite_sites=False, n_pre_snv=60)]


def test_windows_with_copy_numbers(ctx):
    """Copy-number events on a dense table: rejected draws, packed templates, accepted reads counted."""
    from process_amd import _abi as A
    lens = [60_000, 20_000]
    cna = [(0, 0, 5_000, 30_000, 0, A.PSX_CNA_AMP, 2), (0, 1, 1_000, 9_000, 1, A.PSX_CNA_DEL, 0),
           (1, 0, 0, 0, 0, A.PSX_CNA_WGD, 0)]
    w = World(ctx, lens, dict(n_cells=500, n_samples=1, sample_size=90, seed=2), 6e-5, cna=cna)
    for kw in (dict(coverage=400, read_size=150, insert_size_mean=350, insert_size_stddev=10, error_rate=2e-3, purity=0.7),
               dict(coverage=8, read_size=100)):
        a, d, p, n = core.simulate_seq_arrays(ctx, w.g, w.pf, w.pm, 3, **kw)
        oa, od, op, on = O.simulate_seq(w.lens, w.of, w.recs, 3, cna=w.pm.cna(), **kw)
        assert n == on and np.array_equal(d, od) and np.array_equal(a, oa) and np.array_equal(p, op)


AMP, DEL, WGD = 0, 1, 2  # (species, chromosome, start, length, lineage, kind, copies)


@pytest.mark.parametrize("snv", [3e-7, 6e-5])
@pytest.mark.parametrize("cov,ploidy,cna", [
    # a listed window; its edges at a stratum's; more templates in a stratum than the read kernel numbers at a time
    (700.0, 2, [(0, 0, 8192, 8192, 1, AMP, 255), (1, 0, 100, 30_000, 0, DEL, 0), (0, 0, 0, 0, 0, WGD, 0)]),
    # what a listed window does not hold: a 17th event, a fourth doubling, three lineages
    (60.0, 2, [(0, 0, 500 * k, 20_000, k & 1, DEL if k % 5 == 0 else AMP, 1) for k in range(17)]),
    (20.0, 2, [(0, 0, 0, 0, 0, WGD, 0)] * 4),
    (60.0, 3, [(0, 0, 9_000, 20_000, 2, AMP, 2), (1, 1, 0, 4_000, 0, DEL, 0), (1, 0, 0, 0, 0, WGD, 0)]),
    # both lineages gone where every read would start
    (30.0, 2, [(0, 1, 0, 5_000, 0, DEL, 0), (0, 1, 0, 5_000, 1, DEL, 0)])])
def test_copy_number_draws(ctx, snv, cov, ploidy, cna):
    """Counts and reads of segments with copy numbers, sparse and dense tables, with and without a normal share."""
    from process_amd import _abi as A
    kinds = [A.PSX_CNA_AMP, A.PSX_CNA_DEL, A.PSX_CNA_WGD]
    w = World(ctx, [40_000, 5_000], dict(n_cells=500, n_samples=1, sample_size=90, seed=2), snv,
              cna=[(sp, c, at, ln, a, kinds[k], n) for sp, c, at, ln, a, k, n in cna], ploidy=ploidy)
    for kw in (dict(read_size=75, error_rate=2e-3, purity=0.7),
               dict(read_size=100, insert_size_mean=250, insert_size_stddev=10, error_rate=1e-3)):
        kw["coverage"] = cov
        a, d, p, _ = core.simulate_seq_arrays(ctx, w.g, w.pf, w.pm, 3, **kw)
        oa, od, op, on = O.simulate_seq(w.lens, w.of, w.recs, 3, cna=w.pm.cna(), ploidy=ploidy, **kw)
        assert np.array_equal(d, od) and np.array_equal(a, oa) and np.array_equal(p, op)
        rows, m = core.simulate_seq_reads(ctx, w.g, w.pf, w.pm, 3, **kw)
        ref = O.simulate_reads(w.lens, w.g.download(), w.of, w.recs, 3, m, cna=w.pm.cna(), ploidy=ploidy, **kw)
        assert m == on and np.array_equal(rows.numpy()[:m], ref)


@pytest.mark.parametrize("snv", [3e-7, 6e-5])
@pytest.mark.parametrize("cov,ploidy,cna", [
    # draws of the general form with hundreds of copy slots: eight doublings, three lineages, more events than are listed
    (4.0, 2, [(0, 0, 0, 0, 0, WGD, 0)] * 8),
    (8.0, 3, [(0, 1, 0, 9_000, 0, AMP, 255), (0, 1, 0, 9_000, 1, AMP, 255)]),
    (2.0, 2, [(0, 1, 300 * k, 5_000, k & 1, AMP, 255) for k in range(17)])])
def test_copy_number_draws_of_many_slots(ctx, snv, cov, ploidy, cna):
    """A template of the normal genome draws one of the chromosome's copy slots, of which only the first ploidy are its
    copies, however many slots there are: sparse and dense tables, a tumour sample with a normal share and the normal
    sample; the materialised reads are as many."""
    from process_amd import _abi as A
    kinds = [A.PSX_CNA_AMP, A.PSX_CNA_DEL, A.PSX_CNA_WGD]
    w = World(ctx, [40_000, 10_000], dict(n_cells=500, n_samples=1, sample_size=90, seed=2), snv,
              cna=[(sp, c, at, ln, a, kinds[k], n) for sp, c, at, ln, a, k, n in cna], ploidy=ploidy,
              infinite_sites=False, n_pre_snv=6_000 if snv > 1e-6 else 8)
    for kw in (dict(read_size=75, error_rate=2e-3, purity=0.7), dict(read_size=250, insert_size_mean=600,
                                                                    insert_size_stddev=10, purity=0.7)):
        kw["coverage"] = cov
        a, d, p, _ = core.simulate_seq_arrays(ctx, w.g, w.pf, w.pm, 3, **kw)
        oa, od, op, on = O.simulate_seq(w.lens, w.of, w.recs, 3, cna=w.pm.cna(), ploidy=ploidy, **kw)
        assert np.array_equal(d, od) and np.array_equal(a, oa) and np.array_equal(p, op)
        _, m = core.simulate_seq_reads(ctx, w.g, w.pf, w.pm, 3, **kw)
        assert m == on


@pytest.mark.parametrize("kw", [
    # shares of templates with more than three errors below and above the rule; more than eight errors; reads of few bases
    dict(read_size=150, error_rate=3e-3), dict(read_size=250, error_rate=4e-3),
    dict(read_size=150, insert_size_mean=350, insert_size_stddev=10, error_rate=1e-2, purity=0.5),
    dict(read_size=200, error_rate=6e-2), dict(read_size=5, error_rate=0.6)])
@pytest.mark.parametrize("cna", [False, True])
def test_templates_of_many_errors(ctx, kw, cna):
    """Templates whose errors the first draw does not settle, on dense tables: waiting ones counted 48 at a time, the
    last ones of a window, with and without copy numbers."""
    from process_amd import _abi as A
    eng = dict(cna=[(0, 0, 5_000, 30_000, 0, A.PSX_CNA_AMP, 2), (1, 0, 0, 0, 0, A.PSX_CNA_WGD, 0)]) if cna else {}
    w = World(ctx, [60_000, 20_000], dict(n_cells=500, n_samples=1, sample_size=90, seed=2), 2e-4, **eng)
    kw = dict(kw, coverage=150)
    a, d, p, _ = core.simulate_seq_arrays(ctx, w.g, w.pf, w.pm, 3, **kw)
    oa, od, op, _ = O.simulate_seq(w.lens, w.of, w.recs, 3, cna=w.pm.cna(), **kw)
    assert np.array_equal(d, od) and np.array_equal(a, oa) and np.array_equal(p, op) and d.sum() > 0


def test_parts_of_few_strata(ctx):
    """Few strata with many templates: items are cut into parts, in both count kernels and the read kernel."""
    forest = dict(n_cells=300, n_samples=1, sample_size=60, seed=4)
    for snv in (2e-7, 1e-4):
        w = World(ctx, [20_000, 5_000], forest, snv)
        for kw in (dict(coverage=6000, read_size=101, error_rate=5e-3, purity=0.7),
                   dict(coverage=4000, read_size=150, insert_size_mean=350, insert_size_stddev=10, error_rate=1e-3)):
            n = w.check(core.simulate_seq_arrays(ctx, w.g, w.pf, w.pm, 5, **kw)[:3], 5, kw)
            rows, m = core.simulate_seq_reads(ctx, w.g, w.pf, w.pm, 5, **kw)
            assert m == n and np.array_equal(rows.numpy()[:m],
                                             O.simulate_reads(w.lens, w.g.download(), w.of, w.recs, 5, m, **kw))


@pytest.mark.parametrize("n,kw", [
    # few records: reads that wait, some windows' last ones alone; more errors than a lane makes, on either mate
    (300, dict(coverage=150, read_size=100, error_rate=2e-2)),
    (300, dict(coverage=6, read_size=100, error_rate=3e-2)),
    (300, dict(coverage=150, read_size=400, insert_size_mean=900, insert_size_stddev=20, error_rate=3e-2, purity=0.5)),
    # some twenty errors, many of them drawn again
    (300, dict(coverage=40, read_size=40, error_rate=0.5)),
    # more records in a window than are staged, several of them at one position
    (8000, dict(coverage=60, read_size=100, error_rate=0.12)),
    # by windows: templates that wait
    (8000, dict(coverage=60, read_size=250, error_rate=8e-3)),
    (8000, dict(coverage=60, read_size=150, insert_size_mean=350, insert_size_stddev=10, error_rate=6e-3, purity=0.5))])
@pytest.mark.parametrize("cna", [False, True])
def test_reads_of_many_errors(ctx, n, kw, cna):
    """Reads and templates of more than three errors that wait, in both count kernels, with and without copy numbers."""
    from process_amd import _abi as A
    eng = dict(cna=[(0, 0, 5_000, 30_000, 0, A.PSX_CNA_AMP, 2), (1, 0, 0, 0, 0, A.PSX_CNA_WGD, 0)]) if cna else {}
    w = World(ctx, [60_000, 20_000], dict(n_cells=500, n_samples=1, sample_size=90, seed=2), 1e-7, n_pre_snv=n,
              infinite_sites=False, **eng)
    a, d, p, _ = core.simulate_seq_arrays(ctx, w.g, w.pf, w.pm, 3, **kw)
    oa, od, op, _ = O.simulate_seq(w.lens, w.of, w.recs, 3, cna=w.pm.cna(), **kw)
    assert np.array_equal(d, od) and np.array_equal(a, oa) and np.array_equal(p, op) and d.sum() > 0


@pytest.mark.parametrize("snv", [3e-7, 6e-5])
def test_reads_of_chromosomes_with_and_without_events(ctx, snv):
    """The number of reads of a count-only call is that of all its chromosomes, those without copy-number events too:
    the plain call, a batched launch, a plan and a server."""
    from process_amd import _abi as A
    w = World(ctx, [40_000, 30_000, 5_000], dict(n_cells=500, n_samples=2, sample_size=90, seed=2), snv,
              cna=[(0, 1, 2_000, 20_000, 1, A.PSX_CNA_AMP, 2)])
    kw = dict(coverage=30, read_size=75, insert_size_mean=200, insert_size_stddev=8, error_rate=2e-3, purity=0.7)
    on = O.simulate_seq(w.lens, w.of, w.recs, 3, cna=w.pm.cna(), **kw)[3]
    assert core.simulate_seq_arrays(ctx, w.g, w.pf, w.pm, 3, **kw)[3] == on
    assert core.num_reads_table(ctx, w.g, w.pf, w.pm, 3, **kw) == on
    jobs = [core.SeqJob(ctx, w.g, w.pf, w.pm, 3, **kw) for _ in range(2)]
    assert core.simulate_seq_batch(ctx, jobs) == 2 * on
    assert core.SeqPlan(ctx, jobs).run() == 2 * on
    server = core.Server(ctx, 1 << 20)
    assert server.wait(server.submit(w.g, w.pf, w.pm, 3, **kw))[3]["n_reads"] == on
    server.close()


@pytest.mark.parametrize("kw", [
    # windows of four strata and of one; one job's templates wait for their errors; no errors: eight strata
    dict(coverage=2, error_rate=1e-3), dict(coverage=300, error_rate=1e-3, purity=0.5),
    dict(coverage=2, error_rate=2e-2), dict(coverage=300, error_rate=2e-2, purity=0.5), dict(coverage=2)])
@pytest.mark.parametrize("cna", [False, True])
def test_widest_windows(ctx, kw, cna):
    """Mates as far from their reads as the library takes them (4,096 bases): the most bins and the largest bitmap of
    the windows form, 71 KB of LDS."""
    from process_amd import _abi as A
    eng = dict(cna=[(0, 0, 5_000, 30_000, 0, A.PSX_CNA_AMP, 2)]) if cna else {}
    w = World(ctx, [60_000, 9_000, 4_200], dict(n_cells=500, n_samples=1, sample_size=90, seed=2), 1e-7, n_pre_snv=8000,
              infinite_sites=False, **eng)
    kw = dict(kw, read_size=60, insert_size_mean=4000, insert_size_stddev=10)
    a, d, p, n = core.simulate_seq_arrays(ctx, w.g, w.pf, w.pm, 17, **kw)
    oa, od, op, on = O.simulate_seq(w.lens, w.of, w.recs, 17, cna=w.pm.cna(), **kw)
    assert n == on and np.array_equal(d, od) and np.array_equal(a, oa) and np.array_equal(p, op) and d.sum() > 0


@pytest.mark.parametrize("cov,kw", [
    # few templates for the launch's windows: four strata each, two, one
    (0.5, dict(read_size=150, error_rate=3e-2)),
    (0.6, dict(read_size=250, insert_size_mean=600, insert_size_stddev=10, error_rate=8e-3, purity=0.6)),
    (1.0, dict(read_size=150, error_rate=1e-3)),
    (2.0, dict(read_size=150, error_rate=3e-2, purity=0.5)),
    (3.0, dict(read_size=100))])
@pytest.mark.parametrize("n", [300, 20_000, 60_000])
def test_queued_reads_of_several_strata(ctx, n, cov, kw):
    """Windows of queued reads of one, two and four strata in a launch of 600, with few records, with as many as are
    staged of two strata but not of four, and with more than are staged of one."""
    w = World(ctx, [600_000] * 4 + [8_192 + 149, 20_000, 5_000, 400], dict(n_cells=500, n_samples=1, sample_size=90, seed=2),
              1e-8, n_pre_snv=n, infinite_sites=False)
    w.check(core.simulate_seq_arrays(ctx, w.g, w.pf, w.pm, 3, coverage=cov, **kw)[:3], 3, dict(kw, coverage=cov))


def test_autotuner_varies_what_the_jobs_use(ctx):
    """Jobs counted by windows alone leave the block size and the staged records, which that form does not have, at the
    default; with a sparse job every configuration is timed."""
    own = core.Context(0)  # the tuned configuration is the context's
    forest = dict(n_cells=500, n_samples=1, sample_size=90, seed=2)
    kw = dict(coverage=20, read_size=150, insert_size_mean=350, insert_size_stddev=10, error_rate=1e-3)
    dense, sparse = World(own, [300_000], forest, 6e-5), World(own, [300_000], forest, 1e-8)
    for worlds in ([dense], [dense, sparse]):
        jobs = [core.SeqJob(own, w.g, w.pf, w.pm, 3, **kw) for w in worlds]
        cfg, ms = core.autotune(own, jobs)
        assert ms > 0 and cfg.block_threads in (256, 512) and cfg.lds_records in (512, 1024, 2048)
        if worlds == [dense]:
            assert (cfg.block_threads, cfg.lds_records) == (256, 512)
        for w, j in zip(worlds, jobs):
            w.check(j.results(), 3, kw)
