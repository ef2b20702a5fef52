"""Parity of the drop-in kernels (cell list, CSR neighbour list, scan, Morse,
EAM, velocity Verlet, KE/vmax) against the FP64 oracle, through the C-ABI.

Tolerances: integer outputs bit-exact; FP64 forces <= 1e-12 of the RMS
force; mixed forces <= 1e-5 of the RMS force (max over atoms of |dF|).
"""
import ctypes as C

import numpy as np
import pytest

from conftest import GOLDEN, MORSE_CU, force_rel_err, load_golden, system_from_golden
from gpu_helpers import EamTables, csr_build, cell_build, eam_gpu, morse_gpu, say
from oracle import oracle as O
from tdmd_claude_amd import capi
from tdmd_claude_amd import inputs as I
from tdmd_claude_amd.capi import DeviceArray as D

pytestmark = pytest.mark.gpu

FP64, MIXED = capi.TDMD_FP64, capi.TDMD_MIXED
# FP32 pair arithmetic (the reference's mixed contract) on the CSR drop-in
# path: max |dF| over atoms / RMS |F|.
MIXED_TOL = 1e-5


def gas(n, L, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    return rng.uniform(0, 1, size=(n, 3)) * np.asarray(L)


def c1():
    return system_from_golden(load_golden("ref_c1_morse"))


def c2_small():
    s = I.fcc_lattice(8, 8, 8, 3.615)
    I.jitter_uniform(s, 0.02, 4242)
    I.init_velocities(s, 300.0, 42)
    return s


CASES = {
    "c1": lambda: (c1().pos, np.zeros(3), c1().hi, 6.0, 1.0),
    "fcc2048": lambda: (c2_small().pos, np.zeros(3), c2_small().hi, 6.0, 1.0),
    "gas": lambda: (gas(1500, [30.0, 25.0, 28.0], 7), np.zeros(3), np.array([30.0, 25.0, 28.0]),
                    4.0, 0.7),
    "thin": lambda: (gas(300, [14.0, 30.0, 30.0], 3), np.zeros(3), np.array([14.0, 30.0, 30.0]),
                     5.0, 1.0),
}


@pytest.mark.parametrize("case", list(CASES))
def test_cell_list_equals_oracle(case):
    pos, lo, hi, rc, skin = CASES[case]()
    say("cell list", case, len(pos))
    c = cell_build(pos, lo, hi, rc + skin)
    ref = O.cells(pos, lo, hi, rc + skin)
    assert tuple(c["n"]) == ref["n"]
    assert np.array_equal(c["cc"].download(), ref["counts"])
    assert np.array_equal(c["co"].download(), ref["offsets"])
    # within a cell atoms are in index order, as the CPU counting sort leaves them
    assert np.array_equal(c["ca"].download()[:len(pos)], ref["atoms"])


@pytest.mark.parametrize("case", list(CASES))
def test_full_list_bitexact_vs_oracle(case):
    pos, lo, hi, rc, skin = CASES[case]()
    say("csr list", case, len(pos))
    g = csr_build(pos, lo, hi, rc, skin)
    h = O.HalfList(pos, lo, hi, rc, skin)
    rcnt, roff, rnb = h.full()
    cnt = g["counts"].download()
    off = g["offsets"].download()
    nb = g["nbrs"].download()
    assert g["overflow"] == 0
    assert np.array_equal(cnt, rcnt)
    assert np.array_equal(g["counts_pass1"].download(), rcnt)
    assert g["total"] == int(rcnt.sum()) and g["max"] == int(rcnt.max())
    assert np.array_equal(off, np.concatenate([[0], np.cumsum(rcnt)[:-1]]))
    for i in range(len(pos)):
        assert np.array_equal(np.sort(nb[off[i]:off[i] + cnt[i]]), rnb[roff[i]:roff[i] + rcnt[i]])


def rows_reference(pos, lo, hi, periodic, r_list, nc):
    """Rows in the order the list promises: the 27 stencil cells z, y, x outer
    to inner, each cell's atoms by index; d = x_j - x_i in float64, one
    conditional minimum image, r^2 summed unfused."""
    L = hi - lo
    cs = L / np.array(nc)
    c = np.clip(np.trunc((pos - lo) / cs).astype(int), 0, np.array(nc) - 1)
    cell = (c[:, 2] * nc[1] + c[:, 1]) * nc[0] + c[:, 0]
    order = np.argsort(cell, kind="stable")
    start = np.searchsorted(cell[order], np.arange(nc[0] * nc[1] * nc[2] + 1))
    rows = []
    for i in range(len(pos)):
        cand = []
        for dz in (-1, 0, 1):
            for dy in (-1, 0, 1):
                for dx in (-1, 0, 1):
                    n = [(c[i, a] + d) % nc[a] for a, d in enumerate((dx, dy, dz))]
                    k = (n[2] * nc[1] + n[1]) * nc[0] + n[0]
                    cand.append(order[start[k]:start[k + 1]])
        cand = np.concatenate(cand)
        d = pos[cand] - pos[i]
        for a in range(3):
            if periodic[a]:
                x, h = d[:, a].copy(), 0.5 * L[a]
                d[:, a] = np.where(x > h, x - L[a], np.where(x < -h, x + L[a], x))
        r2 = d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1] + d[:, 2] * d[:, 2]
        rows.append(cand[(r2 < r_list * r_list) & (cand != i)])
    return rows


def list_edge_case(name):
    """pos, lo, hi, periodic, r_list, max_neighbors (None: what the count says)."""
    rng = np.random.Generator(np.random.PCG64(11))
    lo = np.array([-3.0, 1.0, 0.5])
    if name == "one":  # a single atom
        return lo + [[1.0, 2.0, 3.0]], lo, lo + 30.0, (1, 1, 1), 4.0, None
    if name == "sparse":  # fewer atoms than cells
        return lo + rng.uniform(0, 40, (200, 3)), lo, lo + 40.0, (1, 1, 1), 4.0, None
    if name == "box of 3 cells below r_list":  # the stencil covers the box
        return lo + rng.uniform(0, 10, (150, 3)), lo, lo + 10.0, (1, 1, 1), 4.9, None
    if name == "cluster":  # cells of hundreds of atoms, stencils beyond one chunk
        p = np.concatenate([rng.normal(15.0, 2.0, (1500, 3)), rng.uniform(0, 30, (500, 3))])
        return lo + np.clip(p, 0, 29.99), lo, lo + 30.0, (1, 1, 1), 4.0, None
    if name == "cut rows":  # capacity below the longest row
        return lo + rng.uniform(0, 14, (900, 3)), lo, lo + 14.0, (1, 1, 1), 4.0, 40
    if name == "outside":  # atoms beyond the faces, some by more than a box
        p = rng.uniform(-6, 18, (700, 3))
        p[::40] += 30.0
        return lo + p, lo, lo + 12.0, (1, 1, 1), 3.9, None
    # open axes, atoms far outside them
    p = rng.uniform(-4, 20, (700, 3))
    p[::50] *= 40.0
    return lo + p, lo, lo + 16.0, (1, 0, 0), 3.9, None


@pytest.mark.parametrize("case", ["one", "sparse", "box of 3 cells below r_list", "cluster",
                                  "cut rows", "outside", "open"])
def test_list_rows_in_order_at_the_edges(case):
    pos, lo, hi, per, r_list, cap = list_edge_case(case)
    pos, hi, N = np.asarray(pos), np.asarray(hi), len(pos)
    say("csr rows", case, N)
    box = capi.Box.make(lo, hi, per)
    n = (C.c_int32 * 3)()
    capi.call("tdmd_cell_grid", C.byref(box), r_list, n, (C.c_double * 3)())
    rows = rows_reference(pos, lo, hi, per, r_list, list(n))
    ncells = n[0] * n[1] * n[2]
    d_pos = D.from_host(np.ascontiguousarray(pos, dtype=np.float64))
    cc, co, ca, ac = D(ncells, np.int32), D(ncells, np.int32), D(N, np.int32), D(N, np.int32)
    wb = C.c_size_t()
    capi.call("tdmd_cell_workspace_bytes", N, ncells, C.byref(wb))
    work = D(wb.value, np.uint8)
    cells = (cc.ptr, co.ptr, ca.ptr, ac.ptr)
    capi.call("tdmd_cell_build", d_pos.ptr, N, C.byref(box), r_list, *cells, work.ptr, None)
    counts, counts2 = D(N, np.int32), D(N, np.int32)
    capi.call("tdmd_nlist_count", d_pos.ptr, N, C.byref(box), r_list, *cells, n, counts.ptr, None)
    want = np.array([len(r) for r in rows])
    assert np.array_equal(counts.download(), want)
    cap = cap or int(want.max())
    offs = np.concatenate([[0], np.cumsum(np.minimum(want, max(cap, 1)))[:-1]]).astype(np.int32)
    d_off, ovf = D.from_host(offs), D(1, np.int32)
    nb = D.from_host(np.full(int(np.minimum(want, cap).sum()) + 64, -7, dtype=np.int32))
    ovf.zero()
    capi.call("tdmd_nlist_fill", d_pos.ptr, N, C.byref(box), r_list, *cells, n, d_off.ptr, nb.ptr,
              counts2.ptr, cap, ovf.ptr, None)
    got = nb.download()
    assert np.array_equal(counts2.download(), want)
    assert int(ovf.download()[0]) == (int(want.max()) if want.max() > cap else 0)
    for i, r in enumerate(rows):
        assert np.array_equal(got[offs[i]:offs[i] + min(len(r), cap)], r[:cap]), i
    assert np.all(got[-64:] == -7)


@pytest.mark.parametrize("n", [1, 255, 4096, 4097, 100000, 1 << 20])
def test_scan_exact(n):
    say("scan", n)
    rng = np.random.Generator(np.random.PCG64(n))
    x = rng.integers(0, 200, size=n).astype(np.int32)
    d_in, d_out, meta = D.from_host(x), D(n, np.int32), D(2, np.int32)
    sb = C.c_size_t()
    capi.call("tdmd_scan_workspace_bytes", n, C.byref(sb))
    w = D(sb.value, np.uint8)
    capi.call("tdmd_scan_exclusive_i32", d_in.ptr, d_out.ptr, n, meta.ptr, w.ptr, None)
    out = d_out.download()
    assert np.array_equal(out, np.concatenate([[0], np.cumsum(x)[:-1]]).astype(np.int32))
    assert list(meta.download()) == [int(x.sum()), int(x.max())]


def morse_oracle(pos, lo, hi, rc, skin):
    h = O.HalfList(pos, lo, hi, rc, skin)
    return O.morse_forces(h, *MORSE_CU)


@pytest.mark.parametrize("case", ["c1", "fcc2048"])
@pytest.mark.parametrize("prec", [FP64, MIXED])
def test_morse_forces_vs_oracle(case, prec):
    pos, lo, hi, rc, skin = CASES[case]()
    say("morse", case, prec)
    g = csr_build(pos, lo, hi, rc, skin)
    f, e = morse_gpu(prec, pos, lo, hi, g, MORSE_CU)
    pe_ref, f_ref = morse_oracle(pos, lo, hi, rc, skin)
    err = force_rel_err(f, f_ref)
    say("  rel force err", err, "pe", e, pe_ref)
    if prec == FP64:
        assert err < 1e-12
        assert e == pytest.approx(pe_ref, rel=1e-12)
    else:
        assert err < MIXED_TOL
        assert e == pytest.approx(pe_ref, rel=1e-6)
    # deterministic energy path: identical on a second call
    f2, e2 = morse_gpu(prec, pos, lo, hi, g, MORSE_CU)
    assert e2 == e and np.array_equal(f2, f)


def test_morse_two_atoms_analytic():
    import json
    ref = json.loads((GOLDEN / "two_atoms_morse_analytic.json").read_text())
    p = ref["potential"]
    pos = np.array([[0.0, 0.0, 0.0], [2.5, 0.0, 0.0]]) + 10.0
    lo, hi = np.zeros(3), np.full(3, 40.0)
    g = csr_build(pos, lo, hi, p["cutoff_A"], 0.5)
    f, e = morse_gpu(FP64, pos, lo, hi, g, (p["D0_eV"], p["alpha_inv_A"], p["r0_A"],
                                             p["cutoff_A"]))
    assert e == pytest.approx(ref["step0"]["U_eV"], rel=1e-14)
    assert f[0, 0] == pytest.approx(ref["step0"]["force_on_atom_1_eV_per_A"][0], rel=1e-14)
    assert f[1, 0] == pytest.approx(ref["step0"]["force_on_atom_2_eV_per_A"][0], rel=1e-14)


def eam_case(pot):
    if pot == "mishin":
        return I.read_setfl(GOLDEN / "Cu_mishin1.eam.alloy")
    return I.johnson_setfl()


@pytest.mark.parametrize("pot", ["mishin", "johnson"])
@pytest.mark.parametrize("prec", [FP64, MIXED])
def test_eam_forces_vs_oracle(pot, prec):
    s = c2_small()
    t = eam_case(pot)
    say("eam", pot, prec)
    tabs = EamTables(prec, t)
    g = csr_build(s.pos, s.lo, s.hi, t.cutoff, 1.0)
    r = eam_gpu(tabs, s.pos, s.types, s.lo, s.hi, g)
    e = O.Eam(tables=t)
    ref = e.forces(O.HalfList(s.pos, s.lo, s.hi, t.cutoff, 1.0), s.types)
    err = force_rel_err(r["forces"], ref["forces"])
    say("  rel force err", err, "pe", r["pe"], ref["pe"])
    say("  rho rel", np.abs(r["rho"] / ref["rho"] - 1).max(), "fp rel",
        np.abs(r["fp"] / ref["fp"] - 1).max())
    if prec == FP64:
        assert err < 1e-12
        assert r["pe"] == pytest.approx(ref["pe"], rel=1e-12)
        assert np.allclose(r["rho"], ref["rho"], rtol=1e-13, atol=0)
        assert np.allclose(r["fp"], ref["fp"], rtol=1e-12, atol=1e-12 * np.abs(ref["fp"]).max())
    else:
        assert err < MIXED_TOL
        assert r["pe"] == pytest.approx(ref["pe"], rel=1e-6)
        assert np.allclose(r["rho"], ref["rho"], rtol=1e-6, atol=0)


def test_eam_multitype_vs_oracle():
    # two synthetic elements with distinct F, rho, phi (the reference's VL-10
    # idea): any type mix-up changes the forces
    base = I.johnson_setfl(nr=2000, nrho=2000)
    p2 = I.JohnsonParams(element="X", E0=3.0, beta=5.0, D_p=0.2, alpha_p=1.4)
    t2 = I.johnson_setfl(p2, nr=2000, nrho=2000)
    r = np.arange(base.nr) * base.dr
    mix = 0.5 * (base.rphi[0] + t2.rphi[0]) * (1.0 + 0.1 * np.exp(-r))
    t = I.SetflTables(["Cu", "X"], [63.546, 50.0], base.nrho, base.drho, base.nr, base.dr,
                      base.cutoff, np.vstack([base.F, t2.F]), np.vstack([base.rho, t2.rho]),
                      np.vstack([base.rphi, mix, t2.rphi]))
    s = c2_small()
    rng = np.random.Generator(np.random.PCG64(1))
    s.types = rng.integers(1, 3, size=s.natoms).astype(np.int32)
    for prec in (FP64, MIXED):
        say("eam multitype", prec)
        r_ = eam_gpu(EamTables(prec, t), s.pos, s.types, s.lo, s.hi,
                     csr_build(s.pos, s.lo, s.hi, t.cutoff, 1.0))
        ref = O.Eam(tables=t).forces(O.HalfList(s.pos, s.lo, s.hi, t.cutoff, 1.0), s.types)
        err = force_rel_err(r_["forces"], ref["forces"])
        say("  rel force err", err)
        assert err < (1e-12 if prec == FP64 else MIXED_TOL)


def cut_rows(natoms, periodic=(1, 1, 1)):
    """The first `natoms` atoms of a jittered crystal with their rows cut to
    lengths around the lane and turn sizes of the row passes (0 slots to all)."""
    s = I.fcc_lattice(8, 8, 8, 3.615)
    I.displace_gaussian(s, 0.05, 77)
    i, j = [], []
    L = s.hi - s.lo
    lengths = [0, 1, 2, 7, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65, 10 ** 6]
    cnt = np.zeros(natoms, dtype=np.int32)
    for a in range(natoms):
        d = s.pos[a] - s.pos
        d -= np.where(periodic, L, 0.0) * np.round(d / L)
        nb = np.nonzero(((d * d).sum(1) < 6.5 ** 2) & (np.arange(s.natoms) != a))[0]
        nb = nb[:lengths[a % len(lengths)]]
        cnt[a] = len(nb)
        i += [a] * len(nb)
        j += list(nb)
    off = np.concatenate([[0], np.cumsum(cnt)[:-1]]).astype(np.int32)
    return s, cnt, off, np.array(i, dtype=np.int64), np.array(j, dtype=np.int32)


@pytest.mark.parametrize("prec", [FP64, MIXED])
@pytest.mark.parametrize("natoms,ntypes,work,per", [(1, 1, True, (1, 1, 1)),
                                                    (129, 1, True, (1, 1, 1)),
                                                    (256, 3, False, (1, 1, 1)),
                                                    (257, 3, True, (1, 0, 1)),
                                                    (1000, 1, None, (1, 1, 1))])
def test_row_passes_at_the_edges(natoms, ntypes, work, per, prec):
    """Morse and EAM over rows of every length class, partial workgroups, one
    and several elements, an open axis; energy by workspace, by atomics and
    absent, against the same sums in numpy float64 (the bounds of the other
    force tests: 1e-12 / 1e-5 of the RMS force)."""
    say("row passes", natoms, ntypes, work, per, prec)
    s, cnt, off, i, j = cut_rows(natoms, per)
    t = I.johnson_setfl(nr=500, nrho=500) if ntypes == 1 else I.johnson_alloy_setfl(nr=500,
                                                                                   nrho=500)
    types = np.random.Generator(np.random.PCG64(5)).integers(1, ntypes + 1, s.natoms)
    L = s.hi - s.lo
    d = s.pos[i] - s.pos[j]
    d -= np.where(per, L, 0.0) * np.round(d / L)
    r = np.sqrt((d * d).sum(1))

    def cubic(v, h, x, deriv):
        a, b, c, dd = O.spline_coeffs(v, h)
        k = np.clip((x / h).astype(int), 0, len(a) - 1)
        y = x - k * h
        return (b[k] + y * (2 * c[k] + 3 * y * dd[k]) if deriv
                else a[k] + y * (b[k] + y * (c[k] + y * dd[k])))

    def pick(tables, which, h, x, deriv=False):  # table which[n] at x[n]
        out = np.zeros(len(x))
        for k in range(len(tables)):
            out[which == k] = cubic(tables[k], h, x[which == k], deriv)
        return out

    rr = np.arange(t.nr) * t.dr
    phi = np.zeros_like(t.rphi)
    phi[:, 1:] = t.rphi[:, 1:] / rr[1:]
    inside = r < t.cutoff
    I_, J_, D_, R_ = i[inside], j[inside], d[inside], r[inside]
    ti, tj = types[I_] - 1, types[J_] - 1
    lo_, hi_ = np.minimum(ti, tj), np.maximum(ti, tj)
    pair = lo_ * ntypes - lo_ * (lo_ + 1) // 2 + hi_
    rho = np.bincount(I_, pick(t.rho, tj, t.dr, R_), natoms)
    fp = np.zeros(s.natoms)  # rows of atoms beyond natoms are empty: rho = 0
    allr = np.concatenate([rho, np.zeros(s.natoms - natoms)])
    fp = pick(t.F, types - 1, t.drho, allr, True)
    f = -(pick(phi, pair, t.dr, R_, True) + fp[I_] * pick(t.rho, tj, t.dr, R_, True)
          + fp[J_] * pick(t.rho, ti, t.dr, R_, True)) / R_
    eam_f = np.stack([np.bincount(I_, f * D_[:, k], natoms) for k in range(3)], 1)
    eam_e = pick(t.F, types[:natoms] - 1, t.drho, rho).sum() + 0.5 * pick(phi, pair, t.dr, R_).sum()
    De, al, r0, rc = MORSE_CU
    inside = r < rc
    e = np.exp(-al * (r - r0))
    w = np.where(inside, -2 * De * al * (1 - e) * e / r, 0.0)
    morse_f = np.stack([np.bincount(i, w * d[:, k], natoms) for k in range(3)], 1)
    morse_e = 0.5 * np.where(inside, De * ((1 - e) ** 2 - 1), 0.0).sum()

    rdt = np.float32 if prec == MIXED else np.float64
    box = capi.Box.make(s.lo, s.hi, per)
    # every atom of the crystal has a row in the arrays (empty beyond natoms),
    # so F'(rho) exists for every neighbour
    M = s.natoms
    cnt_all = np.concatenate([cnt, np.zeros(M - natoms, np.int32)])
    off_all = np.concatenate([off, np.full(M - natoms, len(j), np.int32)])
    d_pos, d_t = D.from_host(s.pos), D.from_host(types.astype(np.int32))
    d_cnt, d_off, d_nb = D.from_host(cnt_all), D.from_host(off_all), D.from_host(np.append(j, np.int32(0)).astype(np.int32))
    tabs = EamTables(prec, t)
    d_rho, d_fp, d_f = D(M, np.float64), D(M, rdt), D((M, 3), rdt)
    d_w = D(M // 256 + 2, np.float64)
    d_e = D.from_host(np.array([2.5]))
    args = (None, None) if work is None else (d_e.ptr, d_w.ptr if work else None)
    tol, etol = (1e-12, 1e-12) if prec == FP64 else (MIXED_TOL, 1e-6)
    scale = max(np.sqrt((eam_f ** 2).sum(1).mean()), 1e-3)
    f0 = pick(t.F, types[natoms:] - 1, t.drho, np.zeros(M - natoms)).sum()
    capi.call("tdmd_eam_compute", tabs.h, d_pos.ptr, d_f.ptr, d_t.ptr, d_nb.ptr, d_off.ptr,
              d_cnt.ptr, M, C.byref(box), d_rho.ptr, d_fp.ptr, *args, None)
    got = d_f.download().astype(np.float64)
    assert np.abs(got[:natoms] - eam_f).max() < tol * scale
    assert np.all(got[natoms:] == 0.0)
    assert np.allclose(d_rho.download()[:natoms], rho, rtol=1e-12 if prec == FP64 else 1e-6)
    if work is not None:
        assert d_e.download()[0] == pytest.approx(2.5 + eam_e + f0, rel=etol)
    # Morse over the first natoms rows only
    d_e = D.from_host(np.array([2.5]))
    args = (None, None) if work is None else (d_e.ptr, d_w.ptr if work else None)
    d_f = D.from_host(np.full((M, 3), 7.0, dtype=rdt))
    p = capi.MorseParams.make(*MORSE_CU)
    capi.call("tdmd_morse_force", prec, d_pos.ptr, d_f.ptr, d_nb.ptr, d_off.ptr, d_cnt.ptr, natoms,
              C.byref(box), C.byref(p), *args, None)
    got = d_f.download().astype(np.float64)
    scale = max(np.sqrt((morse_f ** 2).sum(1).mean()), 1e-3)
    assert np.abs(got[:natoms] - morse_f).max() < tol * scale
    assert np.all(got[natoms:] == 7.0)
    if work is not None:
        assert d_e.download()[0] == pytest.approx(2.5 + morse_e, rel=etol)


@pytest.mark.parametrize("prec", [FP64, MIXED])
def test_velocity_verlet_kernels_vs_oracle(prec):
    s = c1()
    N = s.natoms
    say("vv kernels", prec)
    rng = np.random.Generator(np.random.PCG64(3))
    f = rng.normal(0, 1.0, size=(N, 3))
    rdt = np.float32 if prec == MIXED else np.float64
    f_r = f.astype(rdt).astype(np.float64)  # the force the kernel sees
    masses = s.masses.astype(rdt)
    d_v = D.from_host(s.vel)
    d_x = D.from_host(s.pos)
    d_f = D.from_host(f.astype(rdt))
    d_t = D.from_host(s.types)
    d_m = D.from_host(masses)
    box = capi.Box.make(s.lo, s.hi)
    dt = 0.001
    capi.call("tdmd_half_kick", prec, d_v.ptr, d_f.ptr, d_t.ptr, d_m.ptr, N, dt, None)
    capi.call("tdmd_drift", d_x.ptr, d_v.ptr, N, dt, C.byref(box), None)
    capi.call("tdmd_device_synchronize")
    v = s.vel.copy()
    x = s.pos.copy()
    O.half_kick(v, f_r, s.types, masses.astype(np.float64), dt)
    O.drift(x, v, s.lo, s.hi, dt, single_image=True)
    assert np.allclose(d_v.download(), v, rtol=1e-14, atol=1e-15)
    assert np.allclose(d_x.download(), x, rtol=1e-14, atol=1e-13)
    # fused half kick + drift == half kick then drift (device_velocity_verlet.cu:74-87)
    d_v2 = D.from_host(s.vel)
    d_x2 = D.from_host(s.pos)
    capi.call("tdmd_fused_kick_drift", prec, 0, d_v2.ptr, d_x2.ptr, d_f.ptr, d_t.ptr, d_m.ptr, N,
              dt, C.byref(box), None)
    capi.call("tdmd_device_synchronize")
    assert np.array_equal(d_v2.download(), d_v.download())
    assert np.array_equal(d_x2.download(), d_x.download())


def test_ke_vmax_scale_on_device():
    s = c2_small()
    N = s.natoms
    say("ke/vmax")
    d_v = D.from_host(s.vel)
    d_t = D.from_host(s.types)
    d_m = D.from_host(s.masses)
    wb = C.c_size_t()
    capi.call("tdmd_reduce_workspace_bytes", N, C.byref(wb))
    w = D(wb.value, np.uint8)
    out = D(2, np.float64)
    capi.call("tdmd_compute_ke", FP64, d_v.ptr, d_t.ptr, d_m.ptr, N, out.ptr, w.ptr, None)
    capi.call("tdmd_device_synchronize")
    ke = out.download()[0]
    assert ke == pytest.approx(O.kinetic_energy(s.vel, s.types, s.masses), rel=1e-13)
    capi.call("tdmd_compute_vmax", d_v.ptr, N, out.ptr, w.ptr, None)
    capi.call("tdmd_device_synchronize")
    assert out.download()[0] == pytest.approx(np.sqrt((s.vel ** 2).sum(axis=1)).max(), rel=1e-15)
    capi.call("tdmd_scale_velocities", d_v.ptr, N, 0.5, None)
    capi.call("tdmd_device_synchronize")
    assert np.array_equal(d_v.download(), s.vel * 0.5)


def test_invalid_arguments_return_status():
    box = capi.Box.make((0, 0, 0), (10, 10, 10))
    n = (C.c_int32 * 3)(3, 3, 3)
    st = capi.lib().tdmd_nlist_count(None, 10, C.byref(box), 7.0, None, None, None, None, n,
                                     None, None)
    assert st == 1
    st = capi.lib().tdmd_morse_force(7, None, None, None, None, None, 5, C.byref(box),
                                     C.byref(capi.MorseParams.make(*MORSE_CU)), None, None, None)
    assert st == 1


def test_list_of_a_droplet_with_a_long_cutoff():
    # 2,048 atoms in a box of 1,331 cells: up to ~120 atoms in few cells, whose
    # workgroups are single wavefronts, several to a cell. Rows against the oracle.
    s = I.fcc_lattice(8, 8, 8, 3.615)
    I.jitter_uniform(s, 0.1, 5)
    lo, hi = s.lo, s.lo + 11 * 11.0 + 0.5
    pos = s.pos + 40.0
    say("csr droplet", len(pos))
    g = csr_build(pos, lo, hi, 10.0, 1.0)
    assert g["cells"]["ncells"] == 1331 and g["cells"]["cc"].download().max() > 64
    rcnt, roff, rnb = O.HalfList(pos, lo, hi, 10.0, 1.0).full()
    cnt, off, nb = g["counts"].download(), g["offsets"].download(), g["nbrs"].download()
    assert g["overflow"] == 0
    assert np.array_equal(cnt, rcnt) and np.array_equal(g["counts_pass1"].download(), rcnt)
    for i in range(len(pos)):
        assert np.array_equal(np.sort(nb[off[i]:off[i] + cnt[i]]), rnb[roff[i]:roff[i] + rcnt[i]])
