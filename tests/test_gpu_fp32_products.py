"""The FP32 kernels' products on the bf16 matrix cores (six term products of
the three-term splits, TraitsX6), against FP64 at FP32's own error bound.

One year with the pre-growth endpoint returns the product itself.  With K
terms a destination's value takes ceil(K / 8) roundings of the sum of the
large term products and as many, 2^-8 smaller, of the small ones (each
rounding cut by at most 2^-8 of the last place), one rounding each of the
state, its row's scale, the movement entry and the final sum, and the dropped
term products (three below 2^-25):
|error| <= (ceil(K / 8) (1 + 2^-6) + 6) 2^-24 of a sum of non-negative terms.
A product without any one of the six terms exceeds it."""
import numpy as np
import pytest

from transportoptimiser_amd import landscape as ls
from transportoptimiser_amd import native as nat

pytestmark = pytest.mark.gpu

# Patch counts around the 16-term chunks, the 32-wide tiles and the waves'
# shares.  Alone and in a batch of one road, these path counts leave CUs idle:
# 32-row tiles of eight waves, whole and ragged.
SIZES = [1, 15, 16, 17, 31, 33, 48, 64, 65, 96, 130, 160, 200, 257, 300, 416, 512, 700, 1024]


def _road(P, N, seed):
    rng = np.random.default_rng([seed, P, N])
    # Populations over six decades and entries over nine: every term of the
    # splits, and sums led by one product, count.
    init = 10.0 ** rng.uniform(-3, 3, P)
    trans = 10.0 ** rng.uniform(-9, 0, (P, P))
    trans /= trans.sum(1, keepdims=True)
    surv = 1.0 - rng.uniform(0.0, 0.5, (P, P))
    sd = ls.SpeciesData(trans=np.asfortranarray(trans), surv=np.asfortranarray(surv),
                        init_pop=init, capacity=np.full(P, 1e4), growth=np.zeros(P))
    return ls.RoadProblem([sd], n_years=1, n_paths=N, endpoint=nat.END_PRE_GROWTH, seed=seed)


@pytest.mark.parametrize("N", [1, 70, 256, 300])
def test_one_year_product_within_the_fp32_bound(ctx, N):
    for P in SIZES:
        pr = _road(P, N, 3)
        sd = pr.species[0]
        print(f"P={P} N={N}", flush=True)
        ref = (sd.init_pop[:, None] * sd.trans * sd.surv).sum(0)
        bound = (-(-P // 8) * (1 + 2.0 ** -6) + 6) * 2.0 ** -24
        for out in (ctx.simulate_mte(pr), ctx.simulate_mte_batch([pr], end_pops=True)[0]):
            err = np.abs(out.patch_mean[0] - ref) / ref
            assert err.max() <= bound, (P, err.max(), bound)
            np.testing.assert_allclose(out.end_pops[:, 0], ref.sum(), rtol=bound)


def _filler():
    # 70,000 paths of 20 patches: more workgroups than CUs at any rows, so that
    # every road of the batch takes the tile table's rows.
    return ls.RoadProblem([ls.make_species(np.random.default_rng(81), 20)], n_years=1,
                          n_paths=70000, seed=2, road_id=99)


@pytest.fixture
def keep_tiles(ctx):
    saved = ctx.tile_table(nat.PREC_FP32)
    yield
    for b, t in saved.items():
        ctx.set_tile(nat.PREC_FP32, b, t["rows"], t["split"], t["per_cu"])


# Path counts that make one, two, three, five and seven row tiles (an odd number
# has no 2 x 2 blocks, and a wave's run of tiles crosses row blocks) and whole
# workgroups; rows of 32 to 256, four-wave workgroups (up to 16 output tiles) and
# eight-wave ones (17 to 32).
@pytest.mark.parametrize("rows", [32, 64, 128, 256])
def test_tiles_of_a_full_launch_within_the_fp32_bound(ctx, keep_tiles, rows):
    for b in (128, 256, 512, 1024):
        ctx.set_tile(nat.PREC_FP32, b, min(rows, 32768 // b), 0, 0)
    roads = []
    for P in (1, 17, 48, 64, 96, 128, 130, 200, 256, 300, 416, 512, 700, 1024):
        for N in (32, 70, 150, 220, 256, 300):
            roads.append(_road(P, N, 3))
            roads[-1].road_id = len(roads)
    print(f"{len(roads)} roads at {rows} rows", flush=True)
    batch = ctx.simulate_mte_batch(roads + [_filler()], end_pops=True)
    for pr, out in zip(roads, batch):
        sd, P = pr.species[0], pr.species[0].n_patches
        ref = (sd.init_pop[:, None] * sd.trans * sd.surv).sum(0)
        bound = (-(-P // 8) * (1 + 2.0 ** -6) + 6) * 2.0 ** -24
        err = np.abs(out.patch_mean[0] - ref) / ref
        assert err.max() <= bound, (P, pr.n_paths, err.max(), bound)
        np.testing.assert_allclose(out.end_pops[:, 0], ref.sum(), rtol=bound)
        if rows > 32:  # the same bits as in 32-row tiles, which a road alone takes
            one = ctx.simulate_mte(pr)
            np.testing.assert_array_equal(out.end_pops, one.end_pops)
            np.testing.assert_array_equal(out.patch_mean[0], one.patch_mean[0])


def test_small_launch_takes_fewer_rows_with_the_same_bits(ctx):
    # Alone each road leaves CUs idle and takes 32-row tiles, the smallest with
    # several waves to a tile; with the large one in the batch they take the
    # tile table's rows.
    roads = []
    for i, (P, N) in enumerate([(20, 700), (33, 1000), (100, 1500), (256, 3000), (400, 900)]):
        sp = ls.make_species(np.random.default_rng(70 + i), P)
        roads.append(ls.RoadProblem([sp], n_years=4, n_paths=N, seed=2, road_id=i))
    big = ls.RoadProblem([ls.make_species(np.random.default_rng(80), 64)], n_years=1,
                         n_paths=60000, seed=2, road_id=9)
    print("small roads alone, then in a batch", flush=True)
    alone = [ctx.simulate_mte(r) for r in roads]
    batch = ctx.simulate_mte_batch(roads + [big], end_pops=True)
    for a, b in zip(alone, batch):
        for x, y in ((a.end_pops, b.end_pops), (a.end_mean, b.end_mean), (a.end_sd, b.end_sd),
                     (a.patch_mean[0], b.patch_mean[0]), (a.mte_prob, b.mte_prob)):
            np.testing.assert_array_equal(x, y)


def test_mean_of_nearly_equal_paths_averages_the_roundings(ctx, oracle):
    # REF_CPU's noise is 1e-4 of a population: paths share the first bits of
    # every entry.  A patch's mean over N paths is within the roundings common
    # to all of them (the movement matrix's 2^-24 an entry, averaged over the
    # destination's terms, and the populations' few FP32 constants: 1e-8 rms)
    # and 1 / sqrt(32) of one product's rms error (1.3e-7 at 512 patches): 2.5e-8.
    # Paths that round alike leave 7e-8.
    rng = np.random.default_rng(7)
    sd = ls.make_species(rng, 512)
    pr = ls.RoadProblem([sd], n_years=8, n_paths=1024, growth_law=nat.LAW_REF_CPU, seed=4)
    print("nearly equal paths", flush=True)
    out = ctx.simulate_mte(pr)
    ref = oracle.mte_problem(pr)["patch_mean"][0]
    err = np.linalg.norm(out.patch_mean[0] - ref) / np.linalg.norm(ref)
    assert err <= 4e-8, err


@pytest.mark.parametrize("law", [nat.LAW_LOGNORMAL, nat.LAW_REF_CPU, nat.LAW_REF_GPU])
def test_unchanged_populations_keep_their_exact_total(ctx, law):
    # Nothing moves, dies, grows or varies: a product with the identity adds one
    # exact term to zeros, so every path ends at its initial total exactly and
    # meets a threshold of all of it.
    for P in (1, 20, 100):
        cap = 10.0 + 7.0 * np.arange(P)
        sd = ls.SpeciesData(trans=np.eye(P), surv=np.ones((P, P)), init_pop=3.0 + np.arange(P),
                            capacity=cap, growth=np.zeros(P), params=np.zeros(8), noise_sd=0.0,
                            threshold_ratio=1.0)
        pr = ls.RoadProblem([sd], n_years=5, n_paths=300, growth_law=law)
        print(f"unchanged populations law={law} P={P}", flush=True)
        for out in (ctx.simulate_mte(pr), ctx.simulate_mte_batch([pr], end_pops=True)[0]):
            np.testing.assert_array_equal(out.end_pops[:, 0], sd.init_pop.sum())
            np.testing.assert_array_equal(out.patch_mean[0], sd.init_pop)
            assert out.mte_prob[0] == 1.0


@pytest.mark.parametrize("rows", [64, 256])
def test_scaled_rows_match_oracle_in_any_tile(ctx, oracle, keep_tiles, rows):
    # Jobs with little noise hold their rows scaled: every law, both endpoints,
    # ragged tiles of four and eight waves.  T years carry 3 roundings of 2^-24
    # each beside the product's bound, and the growth's noise constants 1e-6.
    for b in (128, 256, 512, 1024):
        ctx.set_tile(nat.PREC_FP32, b, min(rows, 32768 // b), 0, 0)
    roads, T = [], 6
    for P, N in ((1, 40), (33, 150), (128, 220), (200, 70), (300, 100), (600, 50)):
        for law in (nat.LAW_LOGNORMAL, nat.LAW_REF_CPU, nat.LAW_REF_GPU):
            for end in (nat.END_POST_GROWTH, nat.END_PRE_GROWTH):
                sd = ls.make_species(np.random.default_rng(P), P, noise_sd=0.002)
                roads.append(ls.RoadProblem([sd], n_years=T, n_paths=N, growth_law=law,
                                            endpoint=end, seed=6, road_id=len(roads)))
    print(f"{len(roads)} roads of little noise at {rows} rows", flush=True)
    for pr, out in zip(roads, ctx.simulate_mte_batch(roads + [_filler()], end_pops=True)):
        P = pr.species[0].n_patches
        ref = oracle.mte_problem(pr)
        bound = T * ((-(-P // 8) * (1 + 2.0 ** -6) + 9) * 2.0 ** -24) + 1e-6
        np.testing.assert_allclose(out.end_pops, ref["end_pops"], rtol=bound)
        np.testing.assert_allclose(out.patch_mean[0], ref["patch_mean"][0], rtol=bound)
        one = ctx.simulate_mte(pr)  # 32-row tiles
        np.testing.assert_array_equal(out.end_pops, one.end_pops)
        np.testing.assert_array_equal(out.patch_mean[0], one.patch_mean[0])
