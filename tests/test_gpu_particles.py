"""GPU parity of the particle path: Morton keys, radix sort, bucketing and
active-block compaction against the oracle (all bit-exact: integer work)."""
import numpy as np
import pytest

from msbg_rs_amd import particles as P

pytestmark = pytest.mark.gpu


def oracle_keys(orc, pos):
    pos = np.ascontiguousarray(pos, np.float32)
    keys = np.zeros(pos.shape[0], np.uint32)
    orc.orc_morton_keys(pos, pos.shape[0], keys)
    return keys


def oracle_perm(orc, keys):
    perm = np.zeros(keys.size, np.uint32)
    orc.orc_stable_sort_perm(np.ascontiguousarray(keys, np.uint32), keys.size, perm)
    return perm


def test_morton_keys_match_oracle(hip, orc):
    rng = np.random.default_rng(0)
    pos = rng.uniform(-2.0, 1100.0, size=(100_003, 3)).astype(np.float32)
    pos[:5] = [[0, 0, 0], [1, 0, 0], [0, 1, 0], [0, 0, 1], [1023.5, 1023.5, 1023.5]]
    got = P.morton_keys(pos, lib=hip).get()
    assert np.array_equal(got, oracle_keys(orc, pos))
    assert list(got[:4]) == [0, 1, 2, 4] and got[4] == (1 << 30) - 1


@pytest.mark.parametrize("n", [0, 1, 5, 4095, 4096, 4097, 65537, 1_000_003])
@pytest.mark.parametrize("bits", [30, 32, 12])
def test_radix_sort_is_stable_sort(hip, orc, n, bits):
    rng = np.random.default_rng(n + bits)
    hi = (1 << bits) - 1
    keys = rng.integers(0, hi + 1, size=n, dtype=np.uint64).astype(np.uint32)
    if n > 10:
        keys[::7] = keys[1]  # many duplicates
    vals = np.arange(n, dtype=np.uint32)
    dk, dv = hip.to_device(keys), hip.to_device(vals)
    P.radix_sort_pairs(dk, dv, bits, lib=hip)
    want = oracle_perm(orc, keys)
    assert np.array_equal(dv.get(), want)
    assert np.array_equal(dk.get(), keys[want])


@pytest.mark.parametrize("tiles", [1, 15, 16, 17, 127, 128, 129])
@pytest.mark.parametrize("odd", [0, 1])
def test_radix_tables_about_the_short_scan(hip, orc, tiles, odd):
    """Tables of 256 x tiles digit counts: less than, just and more than a round
    of 4,096 entries, and about the 32,768 that one work-group scans."""
    test_radix_sort_is_stable_sort(hip, orc, 4096 * tiles - odd, 8)


@pytest.mark.parametrize("nb", [(1, 1, 1), (3, 1, 1), (5, 3, 7), (16, 16, 17), (32, 32, 32), (33, 31, 33)])
def test_active_blocks_of_odd_grids(hip, orc, nb):
    """Flags of 1 to 33,759 blocks, most of their counts no multiple of 4."""
    rng = np.random.default_rng(nb[0] + 100 * nb[2])
    s = [16 * k for k in nb]
    pos = (rng.random((200, 3)) * s).astype(np.float32)
    got = P.active_blocks(*s, pos, 4.0, lib=hip)
    lo = np.clip(np.floor(pos / 16 - 0.25).astype(int), 0, None)  # both bounds are exact in float32
    hi = np.minimum(np.trunc(pos / 16 + 0.25).astype(int), np.array(nb) - 1)
    want = {x + nb[0] * (y + nb[1] * z) for l, h in zip(lo, hi) for x in range(l[0], h[0] + 1)
            for y in range(l[1], h[1] + 1) for z in range(l[2], h[2] + 1)}
    assert got.tolist() == sorted(want)


def test_morton_sort_matches_oracle(hip, orc):
    rng = np.random.default_rng(3)
    pos = rng.uniform(0, 512, size=(300_000, 3)).astype(np.float32)
    pos[100:200] = pos[50]  # equal keys keep input order
    keys, perm = P.morton_sort(pos, lib=hip)
    k = oracle_keys(orc, pos)
    want = oracle_perm(orc, k)
    assert np.array_equal(perm.get(), want) and np.array_equal(keys.get(), k[want])


@pytest.mark.parametrize("n,with_mass", [(0, True), (1, True), (4097, False), (300_000, True)])
def test_morton_sort_particles_matches_sort_and_gathers(hip, orc, n, with_mass):
    """The fused sort: keys and permutation as the oracle's stable Morton
    sort, positions / velocities / masses the rows of that permutation (bit
    for bit; masses 1 when none are given)."""
    rng = np.random.default_rng(n + 17)
    pos = rng.uniform(0, 700, size=(n, 3)).astype(np.float32)
    if n > 200:
        pos[100:200] = pos[50]  # equal keys keep input order
    vel = rng.normal(size=(n, 3)).astype(np.float32)
    mass = rng.uniform(0.5, 2.0, n).astype(np.float32) if with_mass else None
    keys, perm, ps, vs, ms = P.morton_sort_particles(pos, vel, mass, lib=hip)
    k = oracle_keys(orc, pos)
    want = oracle_perm(orc, k)
    assert np.array_equal(perm.get(), want) and np.array_equal(keys.get(), k[want])
    assert np.array_equal(ps.get().reshape(n, 3), pos[want])
    assert np.array_equal(vs.get().reshape(n, 3), vel[want])
    assert np.array_equal(ms.get(), mass[want] if with_mass else np.ones(n, np.float32))


@pytest.mark.parametrize("n,nb", [(0, 1), (1, 1), (4, 2), (1000, 64), (10_000, 1024), (1_000_000, 32768),
                                  (200_000, 262144)])
def test_bucket_indices_match_oracle(hip, orc, n, nb):
    rng = np.random.default_rng(n)
    bids = rng.integers(0, nb, n).astype(np.int64)
    if n == 4:
        bids = np.array([1, 0, 1, 0])  # bucket_01
    plan = P.bucket_indices(bids, nb, lib=hip)
    pb, st, perm = plan.host()
    wpb, wst, wperm = orc.bucket_indices(bids, nb)
    assert np.array_equal(pb, wpb) and np.array_equal(st, wst) and np.array_equal(perm, wperm)


def test_particle_bids_match_oracle(hip, orc):
    rng = np.random.default_rng(4)
    pos = rng.uniform(0, [80, 48, 33], size=(50_000, 3)).astype(np.float32)
    got = P.particle_bids(80, 48, 33, pos, lib=hip).get()
    want = np.zeros(pos.shape[0], np.int64)
    orc.orc_particle_bids(80, 48, 33, pos, pos.shape[0], want)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("shape,r_scan,n", [((64, 64, 64), 4.0, 1), ((128, 128, 128), 3.0, 5000),
                                            ((512, 512, 512), 3.0, 200_000), ((32, 48, 16), 4.0, 3)])
def test_active_blocks_match_oracle(hip, orc, shape, r_scan, n):
    rng = np.random.default_rng(n)
    pos = rng.uniform(0, shape, size=(n, 3)).astype(np.float32)
    if n == 3:
        pos = np.array([[17.0, 33.0, 8.0], [0.1, 0.1, 0.1], [31.9, 47.9, 15.9]], np.float32)
    got = P.active_blocks(*shape, pos, r_scan, lib=hip)
    assert np.array_equal(got, orc.active_blocks(*shape, pos, r_scan))


def test_active_blocks_known_answers_on_device(hip):
    assert list(P.active_blocks(64, 64, 64, [[15.5, 8.0, 8.0]], 4.0, lib=hip)) == [0, 1]
    assert list(P.active_blocks(32, 48, 16, [[17.0, 33.0, 8.0]], 4.0, lib=hip)) == [2, 3, 4, 5]
    assert P.active_blocks(64, 64, 64, np.zeros((0, 3), np.float32), 4.0, lib=hip).size == 0


def test_gather_rows(hip):
    rng = np.random.default_rng(5)
    src = rng.normal(size=(1000, 3)).astype(np.float32)
    perm = rng.permutation(1000).astype(np.uint32)
    got = P.gather_rows(hip.to_device(src), hip.to_device(perm), lib=hip).get()
    assert np.array_equal(got, src[perm])


@pytest.mark.parametrize("s", [(80, 80, 80), (64, 64, 128), (320, 320, 640)])
def test_bucket_indices_of_the_upper_z_bound(hip, s):
    """Particles on the upper z bound have ids past the last block, here with a
    bit more than those of 125, 128 and 16,000 blocks: every id once, ascending,
    its particles in input order."""
    nb = [(k + 15) // 16 for k in s]
    rng = np.random.default_rng(s[0])
    pos = rng.uniform(0.0, np.array(s) - 1e-3, (5000, 3)).astype(np.float32)
    pos[::3, 2] = s[2]
    bids = P.particle_bids(*s, pos, lib=hip)
    ids = bids.get()
    n_blocks = nb[0] * nb[1] * nb[2]
    assert int(ids.max()).bit_length() > (n_blocks - 1).bit_length()
    plan = P.bucket_indices(bids, n_blocks, lib=hip)
    blocks, counts = np.unique(ids, return_counts=True)
    pb, starts, perm = plan.host()
    assert np.array_equal(pb, blocks) and np.array_equal(starts, np.concatenate([[0], np.cumsum(counts)]))
    assert np.array_equal(perm, np.argsort(ids, kind="stable"))
