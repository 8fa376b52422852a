"""The mixed form of inversion-symmetric crystals at every padded size: one to seven 32 x 32 tiles per side
in the complex-symmetric exponential (ctem_sym.hip), larger ones in k_sgemm's symmetric products, on bcc Fe and corundum
with Bethe cutoffs that give those beam counts. Against the FP64 form and against the full products (symmetry off):
both are within a few 1e-6 of FP64 at these sizes, the bars are three times that."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# crystal, cutoff, padded sizes that it reaches
SIZES = [("fe", 4.0, {32}), ("fe", 30.0, {32, 64}), ("fe", 60.0, {64}), ("fe", 100.0, {64, 96, 128}), ("fe", 140.0, {96, 128}),
         ("fe", 190.0, {128, 160}), ("fe", 250.0, {160, 192}), ("fe", 320.0, {192, 224, 256}), ("fe", 400.0, {256, 288}),
         ("al2o3", 280.0, {256, 288, 320}), ("al2o3", 400.0, {352, 384, 416, 448}), ("al2o3", 640.0, {512, 544, 576, 608, 640})]


@pytest.mark.parametrize("crystal,weak,sizes", SIZES)
def test_symmetric_exponential_sizes(crystal, weak, sizes):
    from ctemsoft_amd import ebsd, workloads, xtal
    wl = workloads.get({"fe": "fe_c1", "al2o3": "al2o3_c2"}[crystal])
    st, _ = xtal.native_setup(wl.xtal, wl.ekev, wl.dmin, (weak, 2.0 * weak, 0.05))
    if crystal == "al2o3":  # a LUT box over every difference of two list entries, zero outside the reference's
        d = st.lut_dim
        pad = [max(0, int(2 * np.abs(st.hkl[:, a]).max() + st.lut_lo[a])) for a in range(3)]
        lut = np.pad(st.lut.view(np.complex128).reshape(d[2], d[1], d[0]), [(pad[2],) * 2, (pad[1],) * 2, (pad[0],) * 2])
        st = ebsd.Setup(st.hkl, st.ucg.view(np.complex128), st.dbdiff, lut, np.asarray(st.lut_lo) - np.array(pad),
                        st.mlambda, st.dynupz, st.weakcutoff, st.cutoff, st.sgcutoff, st.rmt, st.sites, dsm=st.dsm,
                        isym=st.isym, usehex=st.usehex)
    npx, npy = ebsd.lambert_dims(40, st.usehex)
    ij, k, kn = ebsd.kvectors(npx, npy, st.isym, st.usehex, st.dsm, st.mlambda)
    ctx = ebsd.Context(0)
    ctx.upload_crystal(st)
    lam = np.exp(-np.arange(1, 11) / 8.0).astype(np.float32)
    probe = ctx.plan(k, kn, lam, 1.0, 10.0)
    ns, _ = probe.select()
    probe.close()
    pad = np.maximum(32, (ns + 31) // 32 * 32)
    assert set(pad.tolist()) == sizes
    # of each padded size: the smallest, the largest and a few more
    pick = np.unique(np.concatenate([np.concatenate([i[np.argsort(ns[i], kind="stable")][[0, -1]], i[:4]])
                                     for i in (np.flatnonzero(pad == p) for p in np.unique(pad))]))
    plan = ctx.plan(k[pick], kn[pick], lam, 1.0, 10.0)
    plan.run("fp64")
    ref = plan.dots().copy()
    assert plan.set_symmetry(1)
    plan.run("mixed")
    got = plan.dots().copy()
    assert not plan.set_symmetry(0)
    plan.run("mixed")
    full = plan.dots().copy()
    plan.close()
    ctx.close()
    rel = (np.abs(got - ref) / np.abs(ref)).max(1)
    for p in np.unique(pad[pick]):
        print(f"{crystal} {weak}: npad {p}: {rel[pad[pick] == p].max():.1e}", flush=True)
    assert np.isfinite(got).all() and rel.max() < 1e-5
    assert (np.abs(got - full) / np.abs(ref)).max() < 2e-5


@pytest.mark.parametrize("crystal,ekev,weak,nz,dz", [("fe", 26.8, 17.2, 30, 2.0), ("ni", 26.87, 67.6, 24, 0.5), ("fe", 16.41, 13.5, 53, 1.0),
                                                     ("fe", 20.0, 4.0, 50, 0.5), ("ni", 13.37, 6.5, 46, 1.0)])
def test_few_beams_against_fp64(crystal, ekev, weak, nz, dz):
    """Sets of few beams, where the matrix's 1-norm is nearly its spectral radius and the polynomial's truncation is
    seen in full. Bound: twice what a degree-8 polynomial at the norm 5/4 costs by truncation there (1e-7 to 3e-7), with the
    same again for the 22-bit operands and the FP32 sums."""
    from ctemsoft_amd import ebsd, workloads, xtal
    wl = workloads.get({"fe": "fe_c1", "ni": "ni_c0"}[crystal])
    st, _ = xtal.native_setup(wl.xtal, ekev, wl.dmin, (weak, 2.0 * weak, 0.05))
    npx, npy = ebsd.lambert_dims(25, st.usehex)
    _, k, kn = ebsd.kvectors(npx, npy, st.isym, st.usehex, st.dsm, st.mlambda)
    z = dz * np.arange(1, nz + 1)
    lam = (np.exp(-z / 15.0) / np.exp(-z / 15.0).sum()).astype(np.float32)
    ctx = ebsd.Context(0)
    ctx.upload_crystal(st)
    p = ctx.plan(k, kn, lam, dz, float(max(1, int(nz * dz))))
    ns, _ = p.select()
    p.run("fp64")
    ref = p.dots().copy()
    p.run("mixed")
    err = np.linalg.norm(p.dots() - ref) / np.linalg.norm(ref)
    ctx.close()
    print(f"{crystal} {ekev} kV {weak}: {ns.min()}..{ns.max()} beams, {len(kn)} directions: {err:.2e}", flush=True)
    assert err < 1.2e-6


@pytest.mark.parametrize("weak,npad,count", [(4.0, 32, 3200), (60.0, 64, 1700), (100.0, 96, 700), (140.0, 128, 700), (190.0, 160, 400),
                                             (250.0, 192, 400), (320.0, 224, 400)])
def test_batch_sizes_bitwise(weak, npad, count):
    """More matrices than workgroups (each then walks several, with the same LDS, spill and work buffers) against the same
    directions alone and in small batches, on both sides of where the largest sizes change from a product per launch
    (one and two column blocks a wave) to one launch: the same bits."""
    from ctemsoft_amd import ebsd, workloads, xtal
    wl = workloads.get("fe_c1")
    st, _ = xtal.native_setup(wl.xtal, wl.ekev, wl.dmin, (weak, 2.0 * weak, 0.05))
    npx, npy = ebsd.lambert_dims(40, st.usehex)
    _, k, kn = ebsd.kvectors(npx, npy, st.isym, st.usehex, st.dsm, st.mlambda)
    lam = np.exp(-np.arange(1, 6) / 8.0).astype(np.float32)
    ctx = ebsd.Context(0)
    ctx.upload_crystal(st)

    def dots(i):
        p = ctx.plan(k[i], kn[i], lam, 1.0, 5.0)
        ns, _ = p.select()
        p.run("mixed")
        d = p.dots().copy()
        p.close()
        return ns, d
    ns, _ = dots(np.arange(len(kn)))
    idx = np.flatnonzero(np.maximum(32, (ns + 31) // 32 * 32) == npad)
    assert len(idx) > 70, (npad, ns.min(), ns.max())
    big = np.resize(idx, count)
    _, ref = dots(big)
    assert np.isfinite(ref).all()
    again = ref[len(idx):2 * len(idx)]
    assert np.array_equal(again, ref[:len(again)])
    for n in (1, 3, 12, 13, npad // 4, npad // 4 + 1):
        assert np.array_equal(dots(idx[:n])[1], ref[:n]), n
    ctx.close()
