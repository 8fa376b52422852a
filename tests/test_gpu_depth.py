"""The depth recursion with one wave per matrix (k_depth_wave in ctem_kernels.hip, up to 32 beams in the mixed
forms), over depth counts and numbers of directions that leave its workgroups partly empty: the mixed intensities
against the FP64 form's, to the mixed form's 1e-4 bar, and against the same directions in a large batch, bitwise."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("weak", [1.0, 4.0])
@pytest.mark.parametrize("nz", [1, 2, 7, 50])
def test_wave_depth(weak, nz):
    from ctemsoft_amd import ebsd, workloads, xtal
    wl = workloads.get("fe_c1")
    st, _ = xtal.native_setup(wl.xtal, wl.ekev, wl.dmin, (weak, 2.0 * weak, 0.05))
    npx, npy = ebsd.lambert_dims(20, st.usehex)
    _, k, kn = ebsd.kvectors(npx, npy, st.isym, st.usehex, st.dsm, st.mlambda)
    lam = np.exp(-np.arange(1, nz + 1) / 8.0).astype(np.float32)
    ctx = ebsd.Context(0)
    ctx.upload_crystal(st)

    def dots(m, precision):
        p = ctx.plan(k[:m], kn[:m], lam, 1.0, float(nz))
        ns, _ = p.select()
        p.run(precision)
        d = p.dots().copy()
        p.close()
        return ns, d
    ns, ref = dots(len(kn), "fp64")
    full = dots(len(kn), "mixed")[1]
    assert ns.max() <= 32 and np.isfinite(full).all()
    assert (np.abs(full - ref) / np.abs(ref)).max() < 1e-4
    for m in (1, 2, 3, 5):
        assert np.array_equal(dots(m, "mixed")[1], full[:m])
    ctx.close()
