"""The kernels at the sizes where their work splits change, against the CPU
oracle: contractions beyond one wavefront of primitive pairs, one atom and more
nuclei than lanes, ket lists around the 64-ket blocks, matrices around the
32 x 32 product tiles and the largest size of the row products."""
import numpy as np
import pytest

import oracle

gpu = pytest.mark.gpu
FOCK_TOL = 1e-10


@pytest.fixture(scope="module")
def g():
    import gtfock_amd
    gtfock_amd.lib()
    return gtfock_amd


def _basis(path, nprim):
    """s, p and d shells on hydrogen with the given numbers of primitives."""
    with open(path, "w") as fh:
        fh.write("spherical\n\n****\nH     0\n")
        for l, n in zip("SPD", nprim):
            fh.write("%s   %d   1.00\n" % (l, n))
            for k in range(n):
                fh.write("  %.10f  %.10f\n" % (0.25 * 2.2 ** k, 1.0 / (1 + k)))
        fh.write("****\n")
    return str(path)


def _hydrogens(path, n):
    """n hydrogens in H2 pairs along a folded line (a wide gap, no symmetry)."""
    with open(path, "w") as fh:
        fh.write("%d\n\n" % n)
        for k in range(n):
            x, row = (k // 2) % 24, k // 48
            fh.write("H %.6f %.6f %.6f\n" % (2.3 * x + 0.75 * (k % 2), 2.6 * (row % 8) + 0.05 * x, 2.9 * (row // 8) + 0.03 * (k % 5)))
    return str(path)


# primitives per s, p, d shell; nuclei: 81 primitive pairs and one nucleus,
# the splits between, one primitive and more nuclei than lanes
@gpu
@pytest.mark.parametrize("nprim,natoms", [((9, 5, 2), 1), ((9, 3, 1), 2), ((3, 2, 3), 6), ((1, 1, 1), 66)])
def test_one_electron_edges(g, tmp_path, nprim, natoms):
    gbs, xyz = _basis(tmp_path / "b.gbs", nprim), _hydrogens(tmp_path / "m.xyz", natoms)
    b, ob = g.BasisSet(gbs, xyz), oracle.Basis(gbs, xyz)
    pf = g.PFock(b)
    S, H, Hr = pf.overlap(), pf.core_hamiltonian(), ob.core_hamiltonian()
    pf.close()
    print("one-electron %s %d: %.2e %.2e" % (nprim, natoms, np.abs(S - ob.overlap()).max(), np.abs(H - Hr).max()))
    assert np.abs(S - ob.overlap()).max() < 1e-12
    assert np.abs(H - Hr).max() < 1e-12 * max(10.0, np.abs(Hr).max())


# every order and orientation of the shells; the lanes per quartet follow the
# primitives, from one to all 64 of a wavefront
@gpu
@pytest.mark.parametrize("nprim", [(1, 1, 1), (3, 2, 1), (9, 3, 2)])
def test_quartets_in_every_order(g, tmp_path, nprim):
    gbs, xyz = _basis(tmp_path / "b.gbs", nprim), _hydrogens(tmp_path / "m.xyz", 2)
    b, ob = g.BasisSet(gbs, xyz), oracle.Basis(gbs, xyz)
    erd = g.ERD(b)
    ns = b.nshells
    q = np.array([(M, N, P, Q) for M in range(ns) for N in range(ns) for P in range(ns) for Q in range(ns)], dtype=np.int32)
    worst = 0.0
    for quartet, r in zip(q, erd.quartets(q)):
        ref = ob.eri_quartet(*quartet).reshape(-1)
        worst = max(worst, np.abs(r - ref).max() / max(1.0, np.abs(ref).max()))
    print("quartets %s: %.2e" % (nprim, worst))
    assert worst < 1e-12
    one = erd.quartet(*[int(x) for x in q[-2]])
    assert np.abs(one - ob.eri_quartet(*q[-2]).reshape(-1)).max() < 1e-12 * max(1.0, np.abs(one).max())


# long contractions in every class; STO-3G hydrogens put 55, 66 and 136 kets
# in the (ss| list, around the 64-ket blocks; one and two densities
@gpu
@pytest.mark.parametrize("nprim,natoms", [((9, 5, 2), 1), ((9, 3, 1), 2), ((1, 1, 1), 4),
                                          (None, 2), (None, 10), (None, 11), (None, 16)])
def test_fock_edges(g, sto3g, tmp_path, nprim, natoms):
    gbs = _basis(tmp_path / "b.gbs", nprim) if nprim else sto3g
    xyz = _hydrogens(tmp_path / "m.xyz", natoms)
    b, ob = g.BasisSet(gbs, xyz), oracle.Basis(gbs, xyz)
    rng = np.random.default_rng(77)
    Ds = [0.1 * (a + a.T) for a in rng.normal(size=(2, b.nbf, b.nbf))]
    refs = [sum(ob.fock(D)[:2]) for D in Ds]
    pf = g.PFock(b, tolscr=1e-11, max_numdmat=2)
    err = np.abs(pf.fock(Ds[0]) - refs[0]).max()
    pf.set_num_den_mat(2)
    for k, D in enumerate(Ds):
        pf.put_den_mat(D, index=k)
    pf.commit()
    pf.compute_fock()
    err2 = max(np.abs(pf.get_mat(g.MAT_F, index=k) - refs[k]).max() for k in range(2))
    pf.close()
    print("fock %s %d: %.2e, two densities %.2e" % (nprim, natoms, err, err2))
    assert max(err, err2) < FOCK_TOL


# (dd|dd) holds four components of 16 kets in a wavefront: 1 ket with its 16
# primitive pairs over the lanes, 15, 21 and 36 kets; one density and two
@gpu
@pytest.mark.parametrize("nprim,natoms", [((1, 1, 4), 1), ((1, 1, 2), 5), ((1, 1, 1), 6), ((1, 1, 2), 8)])
def test_fock_dd_lanes(g, tmp_path, nprim, natoms):
    gbs, xyz = _basis(tmp_path / "b.gbs", nprim), _hydrogens(tmp_path / "m.xyz", natoms)
    b, ob = g.BasisSet(gbs, xyz), oracle.Basis(gbs, xyz)
    rng = np.random.default_rng(79)
    Ds = [0.1 * (a + a.T) for a in rng.normal(size=(2, b.nbf, b.nbf))]
    refs = [sum(ob.fock(D)[:2]) for D in Ds]
    pf = g.PFock(b, max_numdmat=2)
    err = np.abs(pf.fock(Ds[0]) - refs[0]).max()
    pf.set_num_den_mat(2)
    for k, D in enumerate(Ds):
        pf.put_den_mat(D, index=k)
    pf.commit()
    pf.compute_fock()
    err2 = max(np.abs(pf.get_mat(g.MAT_F, index=k) - refs[k]).max() for k in range(2))
    pf.close()
    print("fock dd %s %d: %.2e, two densities %.2e" % (nprim, natoms, err, err2))
    assert max(err, err2) < FOCK_TOL


# 1380 functions: the strips of (dd|dd) leave no room for the wavefronts' J_PQ
# buffers in LDS (above 1367), and the class keeps its tiles without them; its
# Schwarz values are 0.67 and 0.15, so a threshold of 0.2 sends a part to FP32
@gpu
@pytest.mark.parametrize("tau", [0.0, 0.2])
def test_fock_without_jpq_buffers(g, tmp_path, tau):
    gbs, xyz = str(tmp_path / "b.gbs"), str(tmp_path / "m.xyz")
    with open(gbs, "w") as fh:
        fh.write("spherical\n\n****\nH     0\nS   1   1.00\n  0.75  1.0\nD   1   1.00\n  0.75  1.0\n****\n")
    with open(xyz, "w") as fh:
        fh.write("230\n\n")
        for k in range(230):
            i = k // 2
            fh.write("H %.6f %.6f %.6f\n" % (9.0 * (i % 5) + 0.75 * (k % 2), 9.0 * (i // 5 % 5) + 0.1 * (i % 3), 9.0 * (i // 25)))
    b, ob = g.BasisSet(gbs, xyz), oracle.Basis(gbs, xyz)
    assert b.nbf == 1380
    a = np.random.default_rng(78).normal(size=(b.nbf, b.nbf))
    D = 0.1 * (a + a.T)
    pf = g.PFock(b)
    pf.set_precision(tau)
    kernel = pf.class_kernel(20)
    err = np.abs(pf.fock(D) - sum(ob.fock(D)[:2])).max()
    low = pf.mixed_counts()[0][20]
    pf.close()
    print("fock 1380, tau %g: %s, %d quartets in FP32, %.2e" % (tau, kernel, low, err))
    assert kernel.startswith("eri_jk_tile_kernel<2, 2, 2, 2,")
    if tau == 0.0:
        assert err < FOCK_TOL
    else:
        # an integral below tau is off by the FP32 rounding of about 16 sums;
        # a Fock element adds up to n^2 of them, with errors of either sign
        assert low > 0 and err < 16 * 2.0**-24 * tau * b.nbf * np.abs(D).max()


# Hermite coefficients of a primitive pair, all and structural nonzeros
FULL = {"ss": 1, "ps": 12, "pp": 90, "ds": 50, "dp": 300, "dd": 875}
NONZERO = {"ss": 1, "ps": 6, "pp": 33, "ds": 24, "dp": 122, "dd": 391}


def _prim_pairs(nprim, natoms):
    """{pair type: primitive pairs} of natoms atoms that each have an s, a p and a
    d shell of nprim primitives."""
    out = {}
    for t in FULL:
        a, b = ("spd".index(c) for c in t)
        out[t] = (natoms * (natoms + 1) // 2 if a == b else natoms * natoms) * nprim[a] * nprim[b]
    return out


# the molecules of a batch share the 64-ket blocks of the records: one molecule's
# lists of 1 to 3 kets pad 64, sixty-four of them a few in a hundred
@gpu
def test_batch_memory_shares_ket_blocks(g, tmp_path):
    nprim, natoms, nmol = (6, 3, 1), 2, 64
    gbs, xyz = _basis(tmp_path / "b.gbs", nprim), _hydrogens(tmp_path / "m.xyz", natoms)
    bases = [g.BasisSet(gbs, xyz) for _ in range(nmol)]
    one, many = g.Batch(bases[:1]), g.Batch(bases)
    used1, used = one.stats()["device_bytes"], many.stats()["device_bytes"]
    one.close()
    many.close()
    # p, P, bound and both coefficient forms; the record with, for pp, ds and
    # dp, the full form; a quarter more where a block mixes primitive counts
    pairs = sum(n * (40 + 8 * (FULL[t] + NONZERO[t])
                     + 1.25 * (8 + 16 * (2 + (NONZERO[t] + 1) // 2) + (8 * FULL[t] if t in ("pp", "ds", "dp") else 0)))
                for t, n in _prim_pairs(nprim, natoms).items())
    print("one %.2f MB, %d %.2f MB, a molecule's primitive pairs %.3f MB" % (used1 / 1e6, nmol, used / 1e6, pairs / 1e6))
    # beside them what one holds at most, and 32 KB a molecule for lists, tiles
    # and matrices
    assert used < used1 + nmol * (pairs + 32768)


# without d functions nothing reads the full coefficients of the kets: the
# primitive pairs, a record each, and a tenth for padded blocks (300 kets in 320
# places), lists, tiles
@gpu
def test_memory_without_d_functions(g, tmp_path):
    nprim, natoms = (4, 4, 1), 24
    gbs = _basis(tmp_path / "b.gbs", nprim)
    with open(gbs) as fh:
        text = fh.read()
    with open(gbs, "w") as fh:
        fh.write(text[:text.index("D   1")] + "****\n")
    pf = g.PFock(g.BasisSet(gbs, _hydrogens(tmp_path / "m.xyz", natoms)))
    used = pf.stats()["device_bytes"]
    pf.close()
    pairs = sum(n * (40 + 8 * (FULL[t] + NONZERO[t]) + 8 + 16 * (2 + (NONZERO[t] + 1) // 2))
                for t, n in _prim_pairs(nprim, natoms).items() if "d" not in t)
    print("device memory %.1f MB, primitive pairs %.1f MB" % (used / 1e6, pairs / 1e6))
    assert used < 1.1 * pairs + 0.3e6  # Boys tables


# the FP32 tiles add a rounded copy of the nonzero coefficients, and lists of a
# quarter of it at most (a run of 64 kets has 20 bytes)
@gpu
def test_mixed_precision_memory(g, tmp_path):
    nprim, natoms = (4, 4, 4), 20
    b = g.BasisSet(_basis(tmp_path / "b.gbs", nprim), _hydrogens(tmp_path / "m.xyz", natoms))
    pf = g.PFock(b)
    before = pf.stats()["device_bytes"]
    pf.set_precision(1e-4)
    added = pf.stats()["device_bytes"] - before
    pf.close()
    copy = sum(4 * NONZERO[t] * n for t, n in _prim_pairs(nprim, natoms).items())
    print("FP64 %.1f MB, mixed adds %.1f MB, coefficients %.1f MB" % (before / 1e6, added / 1e6, copy / 1e6))
    assert added < 1.25 * copy


# the server admits jobs by this estimate: it covers what a batch of the molecule
# allocates, and not 40 % more, or a budget holds fewer jobs than it could
@gpu
@pytest.mark.parametrize("mol", ["c10h22", "c54h18"])
def test_job_estimate_is_close(g, gbs, mol_dir, mol):
    b = g.BasisSet(gbs, str(mol_dir / (mol + ".xyz")))
    est = g.lib().gtf_batch_job_bytes(b.h)
    bt = g.Batch([b], tau=1e-4)
    bt.set_purif_precision("split")
    bt.scf_begin(max_iters=3)
    bt.scf_step()
    bt.scf_step()
    used = bt.stats()["device_bytes"]
    bt.close()
    print("%s: estimate %.1f MB, allocated %.1f MB" % (mol, est / 1e6, used / 1e6))
    assert used <= est <= 1.4 * used


# the kernel named is the one launched: (dd|dd) stages the Boys table and ten
# density rows in LDS (160 KB) beside its ten exchange rows up to 521 functions
@gpu
@pytest.mark.parametrize("natoms,staged", [(86, "true"), (88, "false")])
def test_class_kernel_names_the_staging(g, tmp_path, natoms, staged):
    gbs = str(tmp_path / "b.gbs")
    with open(gbs, "w") as fh:
        fh.write("spherical\n\n****\nH     0\nS   1   1.00\n  0.75  1.0\nD   1   1.00\n  0.75  1.0\n****\n")
    b = g.BasisSet(gbs, _hydrogens(tmp_path / "m.xyz", natoms))
    assert b.nbf == 6 * natoms
    pf = g.PFock(b)
    assert pf.tile_shape(20)["boys_lds"] == 1
    assert pf.class_kernel(20) == "eri_jk_tile_kernel<2, 2, 2, 2, 1, double, %s>" % staged
    pf.close()


# one tile, a remainder of two, exact tiles, several tiles
@gpu
@pytest.mark.parametrize("n", [2, 32, 34, 64, 66, 130])
def test_purification_edges(g, sto3g, tmp_path, n):
    xyz = _hydrogens(tmp_path / "m.xyz", n)
    b, ob = g.BasisSet(sto3g, xyz), oracle.Basis(sto3g, xyz)
    S = ob.overlap()
    X = oracle.inv_sqrt(S)
    F = X @ ob.core_hamiltonian() @ X
    F = 0.5 * (F + F.T)
    Dref, _ = oracle.purification(F, X, ob.nocc)
    pu = g.Purif(b)
    pu.set_xs(X, S)
    D, _ = pu.purify(F)
    pu.close()
    print("purification n = %d: %.2e" % (n, np.abs(D - Dref).max()))
    assert np.abs(D - Dref).max() < 1e-10


# A B^T: below, at and above a tile, and both sides of the largest size of the
# row products; each element within the rounding of its sum of k products
@gpu
@pytest.mark.parametrize("n", [1, 31, 33, 64, 100, 511, 512, 513])
def test_dgemm_edges(g, n):
    rng = np.random.default_rng(n)
    A, B = rng.normal(size=(2, n, n))
    bound = 2.0 * (n + 1) * np.finfo(float).eps * (np.abs(A) @ np.abs(B.T)) + 1e-300
    assert (np.abs(g.dgemm(A, B, transB=True) - A @ B.T) <= bound).all()


# a molecule's products are those of its own size, whatever shares the batch:
# 36 functions alone and beside 258 and 516 (the matrices are padded to a
# multiple of 64; the row products end at 512).  The regrouped batch carries S,
# H and X over, and the first build is of a zero density, so its results are exact.
@gpu
@pytest.mark.parametrize("large", [43, 86])
def test_batch_products_do_not_depend_on_the_batch(g, tmp_path, large):
    gbs = _basis(tmp_path / "b.gbs", (2, 2, 2))
    with open(gbs) as fh:
        text = fh.read()
    with open(gbs, "w") as fh:  # s and d: six functions an atom
        fh.write(text[:text.index("P   2")] + text[text.index("D   2"):])
    small = g.BasisSet(gbs, _hydrogens(tmp_path / "s.xyz", 6))
    big = g.BasisSet(gbs, _hydrogens(tmp_path / "l.xyz", large))
    assert (small.nbf, big.nbf) == (36, 6 * large)
    alone = g.Batch([small])
    alone.scf_begin(max_iters=3)
    beside, origin = alone.regroup([big])
    assert list(origin) == [0, -1]
    alone.scf_step()
    beside.scf_step()
    D, E = alone.get_density()[0], beside.get_density()[0]
    alone.close()
    beside.close()
    assert np.abs(D).max() > 0.1
    assert np.array_equal(D, E)


# the symmetric update of the split products: one tile, remainders, several
# tiles; the last iterations are FP64, so the projector is as exact as theirs
@gpu
@pytest.mark.parametrize("n", [2, 34, 64, 130])
def test_split_purification_edges(g, sto3g, tmp_path, n):
    xyz = _hydrogens(tmp_path / "m.xyz", n)
    b, ob = g.BasisSet(sto3g, xyz), oracle.Basis(sto3g, xyz)
    S = ob.overlap()
    X = oracle.inv_sqrt(S)
    pu = g.Purif(b)
    pu.set_xs(X, S)
    pu.set_precision("split")
    D, _ = pu.purify(X @ ob.core_hamiltonian() @ X)
    pu.close()
    print("split n = %d: %.2e %.2e" % (n, np.abs(D - D.T).max(), np.abs(D @ S @ D - D).max()))
    assert np.abs(D - D.T).max() < 1e-12
    assert np.abs(D @ S @ D - D).max() < 1e-10
    assert abs(np.trace(D @ S) - ob.nocc) < 1e-9
