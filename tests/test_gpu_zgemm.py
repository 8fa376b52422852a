"""The batched complex FP64 product (k_zgemm, k_zgemm_few in ctem_kernels.hip) through the entries built on
it, at sizes around its 16-, 32- and 64-wide tiles. One matrix (few tiles): CalcLgh3 against scipy's
exponential; both evaluate exp to the last digits of doubles and the depth recursion adds a few roundings
a step, so 1e-11 of the largest entry bounds it with two digits to spare. Many matrices and the pair product:
the adjoint of all directions at once against the sum over small groups, which take the other kernel; only the
order of the sum over directions differs."""
import numpy as np
import pytest
import scipy.linalg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 15, 16, 17, 32, 33, 63, 65, 100, 129, 224])
def test_one_matrix(n):
    from ctemsoft_amd import ebsd
    rng = np.random.default_rng(n)
    d = 0.3 * (rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))) / np.sqrt(n) + 0.02j * np.eye(n)
    thick, kn, dz, nz = 9.0, 2.5, 1.0, 9
    lam = np.exp(-np.arange(1, nz + 1) / 6.0).astype(np.float32)  # the entry takes the weights in single precision
    ctx = ebsd.Context(0)
    got = ctx.calclgh3(d, thick, kn, dz, lam)
    ctx.close()
    e = scipy.linalg.expm(2j * np.pi * dz / float(np.float32(2.0 * kn)) * d)
    psi = [e[:, 0]]
    for _ in range(nz - 1):
        psi.append(e @ psi[-1])
    psi = np.array(psi).T
    want = dz / thick * (psi * lam) @ psi.conj().T
    err = np.abs(np.asarray(got) - want).max() / np.abs(want).max()
    print(f"n {n}: {err:.1e}", flush=True)
    assert err < 1e-11


@pytest.mark.parametrize("weak,nz", [(20.0, 1), (60.0, 13), (140.0, 8), (240.0, 20)])
def test_groups_of_directions(weak, nz):
    from ctemsoft_amd import ebsd, workloads, xtal
    wl = workloads.get("fe_c1")
    st, _ = xtal.native_setup(wl.xtal, wl.ekev, wl.dmin, (weak, 2.0 * weak, 0.05))
    npx, npy = ebsd.lambert_dims(30, st.usehex)
    _, k, kn = ebsd.kvectors(npx, npy, st.isym, st.usehex, st.dsm, st.mlambda)
    k, kn = k[:300], kn[:300]
    lam = np.exp(-np.arange(1, nz + 1) / 8.0).astype(np.float32)
    rng = np.random.default_rng(5)
    w = rng.standard_normal((len(kn), 1))
    ctx = ebsd.Context(0)
    ctx.upload_crystal(st)

    def grad(a, b):
        p = ctx.plan(k[a:b], kn[a:b], lam, 1.0, float(nz))
        ns, _ = p.select()
        g, gb = p.adjoint(w[a:b])
        p.close()
        return ns, g, gb
    ns, g, gb = grad(0, len(kn))
    parts = [grad(a, a + 15) for a in range(0, len(kn), 15)]
    ctx.close()
    print(f"{weak}: {ns.min()}..{ns.max()} beams, {len(kn)} directions", flush=True)
    scale = sum(np.abs(p[1]).max() for p in parts)
    assert np.abs(g - sum(p[1] for p in parts)).max() <= 1e-12 * scale
    assert np.abs(gb - sum(p[2] for p in parts)).max() <= 1e-12 * sum(np.abs(p[2]).max() for p in parts)
