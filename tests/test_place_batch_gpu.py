"""Batched placement (psx_place_mutations_batch): many forests over one
genome in one call, each table byte for byte the single-forest placement's
and the oracle's, with the infinite-sites model on and off, ID signatures,
copy-number drivers, a coarse context sampling, an empty table, jobs whose
redraw rounds outlast the others' and many tiny jobs sharing waves; a bad job
fails the batch with its index in the message."""
from __future__ import annotations

import numpy as np
import pytest

import cases
from oracle import oracle as O
from process_amd import _abi as A
from process_amd import core
from process_amd._lib import PsxError

pytestmark = pytest.mark.gpu

LENS = [400_000, 150_000, 60_000]


def forests(ctx, specs):
    out = []
    for n_cells, seed, two in specs:
        fd = cases.forest(n_cells=n_cells, n_samples=2, sample_size=min(100, n_cells // 4), seed=seed,
                          two_species=two)
        f = core.Forest(ctx, fd["cell_id"], fd["parent"], fd["species"], fd["sample"], fd["birth"], fd["n_samples"])
        of = O.Forest(fd["cell_id"], fd["parent"], fd["species"], fd["sample"], fd["birth"], fd["n_samples"])
        out.append((f, of, two))
    return out


def engines(packed, fs):
    rng = np.random.default_rng(4)
    ids = rng.dirichlet(np.ones(A.PSX_ID_CLASSES), size=2)
    e = []
    for k, (_, _, two) in enumerate(fs):
        if two:
            eng = cases.engine(packed, LENS, snv=(1 + k) * 4e-7, indel=1e-7, pre_snv=3 * k, pre_indel=k,
                               infinite_sites=k != 2)
        else:
            sig = cases.signatures(1, k)
            eng = dict(snv_rate=[6e-7], indel_rate=[5e-8], sbs=sig, epoch_start=[0.0], exposure=[[1.0]],
                       n_pre_snv=2, n_pre_indel=0, pre_sbs=0, indel_max_len=10, indel_len_p=0.5,
                       infinite_sites=True, ploidy=2, drivers=[], germline=[])
        e.append(eng)
    e[1].update(id_sig=ids, id_exposure=[[0.3, 0.7], [0.6, 0.4]], pre_id=1)
    e[3]["context_sampling"] = 20
    e[4]["cna"] = [(1, 0, 1000, 20_000, 0, A.PSX_CNA_AMP, 2), (1, 0, 0, 0, 0, A.PSX_CNA_WGD, 0)]
    # an empty table: no rates, no drivers, no germline, no preneoplastic mutations
    e[5].update(snv_rate=[0.0], indel_rate=[0.0], n_pre_snv=0)
    # dense: about one mutation per 60 bases, many more redraw rounds than the other jobs
    e[6].update(snv_rate=[3e-5, 3e-5], indel_rate=[3e-6, 3e-6])
    return e


def test_batch_equals_single_and_oracle(ctx):
    g = core.Genome(ctx, LENS, seed=13)
    packed = g.download()
    specs = [(800, 1, True), (1200, 2, True), (600, 3, True), (900, 4, True), (700, 5, True), (300, 6, False),
             (1000, 7, True)]
    fs = forests(ctx, specs)
    es = engines(packed, fs)
    seeds = [101 + 7 * k for k in range(len(fs))]
    batch = core.Mutations.place_batch(ctx, g, [f for f, _, _ in fs], seeds, es)
    assert len(batch) == len(fs)
    for k, ((f, of, _), eng, sd) in enumerate(zip(fs, es, seeds)):
        got = batch[k].download()
        one = core.Mutations.place(ctx, g, f, sd, **eng)
        assert got.tobytes() == one.download().tobytes(), k
        assert np.array_equal(batch[k].cna(), one.cna()), k
        assert got.tobytes() == O.place_mutations(LENS, packed, of, sd, **eng).tobytes(), k
    assert batch[5].n == 0
    assert batch[6].n > 5 * batch[0].n
    # the tables share one block: freeing some leaves the others whole
    keep = batch[6].download()
    for k in range(6):
        batch[k].close()
    assert batch[6].download().tobytes() == keep.tobytes()


def test_batch_error_names_the_job(ctx):
    g = core.Genome(ctx, LENS, seed=13)
    packed = g.download()
    fs = forests(ctx, [(400, 1, True), (400, 2, True), (400, 3, True)])
    es = [cases.engine(packed, LENS) for _ in fs]
    pos = es[2]["drivers"][0][2]
    base = cases.base_of(packed, LENS, 0, pos)
    es[2]["drivers"] = [(1, 0, pos, base, -1)]  # alternative equal to the reference base
    with pytest.raises(PsxError, match="job 2: invalid driver 0"):
        core.Mutations.place_batch(ctx, g, [f for f, _, _ in fs], [1, 2, 3], es)
    es[2] = cases.engine(packed, LENS)
    es[0]["ploidy"] = 0
    with pytest.raises(PsxError, match="job 0: invalid ploidy"):
        core.Mutations.place_batch(ctx, g, [f for f, _, _ in fs], [1, 2, 3], es)


def test_many_tiny_jobs_share_waves(ctx):
    """48 forests of 12-60 cells: each job has a few to tens of mutations and
    nodes, so most waves of every per-node and per-mutation kernel hold
    several jobs (one pass per job in the wave); every table equals the
    single-forest placement, and every eighth the oracle's."""
    g = core.Genome(ctx, LENS, seed=21)
    packed = g.download()
    rng = np.random.default_rng(9)
    fs, es, seeds = [], [], []
    for k in range(48):
        n = int(rng.integers(12, 61))
        fd = cases.forest(n_cells=n, n_samples=1, sample_size=max(2, n // 4), seed=100 + k)
        f = core.Forest(ctx, fd["cell_id"], fd["parent"], fd["species"], fd["sample"], fd["birth"], fd["n_samples"])
        of = O.Forest(fd["cell_id"], fd["parent"], fd["species"], fd["sample"], fd["birth"], fd["n_samples"])
        fs.append((f, of))
        es.append(cases.engine(packed, LENS, snv=float(rng.uniform(2e-6, 2e-5)), indel=2e-7, drivers=k % 3 == 0,
                               germline=k % 4 == 0, infinite_sites=k % 5 != 0))
        seeds.append(500 + k)
    batch = core.Mutations.place_batch(ctx, g, [f for f, _ in fs], seeds, es)
    sizes = []
    for k, ((f, of), eng, sd) in enumerate(zip(fs, es, seeds)):
        got = batch[k].download()
        sizes.append(len(got))
        assert got.tobytes() == core.Mutations.place(ctx, g, f, sd, **eng).download().tobytes(), k
        if k % 8 == 0:
            assert got.tobytes() == O.place_mutations(LENS, packed, of, sd, **eng).tobytes(), k
    assert sum(sizes) > 48 * 5 and min(sizes) < 64


def test_tables_in_blocks_used_before(ctx):
    """A table's memory goes to a later table: sizes that fit an idle block and sizes that do not, tables freed in any
    order, from two threads with a context each and from a third context's; every table is the oracle's."""
    import threading
    g = core.Genome(ctx, LENS, seed=5)
    packed = g.download()
    fs = forests(ctx, [(400, 1, True), (900, 2, True)])
    rates = [1e-6, 1.2e-6, 5e-6, 2e-5]
    want = {}
    for k, (f, of, _) in enumerate(fs):
        for r in rates:
            want[k, r] = O.place_mutations(LENS, packed, of, 9, **cases.engine(packed, LENS, snv=r)).tobytes()
    errors = []

    def work(seed, own):
        try:
            c = core.Context(0) if own else ctx
            gc = core.Genome(c, LENS, packed=packed)
            rng = np.random.default_rng(seed)
            held = []
            for _ in range(24):
                k, r = int(rng.integers(2)), rates[int(rng.integers(4))]
                m = core.Mutations.place(c, gc, fs[k][0], 9, **cases.engine(packed, LENS, snv=r))
                held.append((m, want[k, r]))
                if len(held) > 3:
                    m, w = held.pop(int(rng.integers(4)))
                    assert m.download().tobytes() == w
                    m.close()
            for m, w in held:
                assert m.download().tobytes() == w
        except Exception as e:  # reported by the caller's thread
            errors.append(e)

    ts = [threading.Thread(target=work, args=(s, True)) for s in (1, 2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    work(3, False)
    assert not errors, errors


@pytest.mark.parametrize("lens,share,pre,infinite", [
    ([400_000], 1.0, 1024, True), ([400_000], 1.0, 1025, True),  # one launch of the library; the bucket sort
    ([700_000, 90_000, 37], 1.0, 6000, True),                    # a chromosome shorter than a bucket
    ([3000], 1.0, 3000, False),                                  # several mutations at every position
    ([2_000_000], 0.004, 5000, False),                           # all in 8 kb: a bucket overfilled, sorted by radix
    ([2_000_000], 0.0008, 1900, False),                          # a bucket's entries in few of its parts
    ([2_000_000], 1e-5, 1500, False)])                           # at 20 positions
def test_order_of_crowded_tables(ctx, lens, share, pre, infinite):
    """The bucket sort of the first attempts over table sizes and densities, alone and in a batch: mutations confined to
    the first bases of a reference that is one letter elsewhere."""
    rng = np.random.default_rng(7)
    seqs = []
    for k, n in enumerate(lens):
        s = np.full(n, "A")
        m = int(n * share)
        s[:m] = rng.choice(list("CG") if share < 1.0 else list("ACGT"), m)
        seqs.append("".join(s))
    import process_amd as pa
    names = [str(k + 1) for k in range(len(lens))]
    ref = pa.ReferenceGenome(dict(zip(names, lens)), sequences=dict(zip(names, seqs)))
    packed = ref.packed
    g = core.Genome(ctx, ref.lengths, packed=packed)
    sbs = np.zeros((1, 96))
    sbs[0, :48] = 1.0 / 48  # C>N
    if share < 1.0:  # of C and G neighbours only
        sbs[0] = 0.0
        for sub in range(3):
            for five in (1, 2):
                for three in (1, 2):
                    sbs[0, sub * 16 + five * 4 + three] = 1.0 / 12
    fs, es = forests(ctx, [(300, 4, False), (200, 5, False)]), []
    for k in range(2):
        es.append(dict(snv_rate=[1e-9], indel_rate=[0.0], sbs=sbs, epoch_start=[0.0], exposure=[[1.0]],
                       n_pre_snv=pre >> k, n_pre_indel=0, pre_sbs=0, indel_max_len=10, indel_len_p=0.5,
                       infinite_sites=infinite, ploidy=2, drivers=[], germline=[]))
    want = [O.place_mutations(ref.lengths, packed, of, 3 + k, **es[k]).tobytes() for k, (_, of, _) in enumerate(fs)]
    batch = core.Mutations.place_batch(ctx, g, [f for f, _, _ in fs], [3, 4], es)
    for k, (f, of, _) in enumerate(fs):
        assert batch[k].download().tobytes() == want[k], k
        assert core.Mutations.place(ctx, g, f, 3 + k, **es[k]).download().tobytes() == want[k], k
