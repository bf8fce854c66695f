"""Multigrid level operators that form their geometric factors from the element
corners (mgGeometry = 1, the default, on meshes of trilinear elements) against
the same operators streaming the stored factors (mgGeometry = 0, the
reference's way): every level's A x agrees to 1e-13 relative in FP64 and 1e-5 in
FP32 (there the stored factors are FP64 values rounded once, the formed ones
FP32 arithmetic throughout), at orders 1..9, Poisson and Helmholtz, on the
Kershaw box and a .re2 box with rotated elements; on a curved (sine-mapped)
box the option changes nothing (bit for bit); and full p-MG solves take the
same iterations (+-1) to the same solution (1e-8)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def handles(gpu, mesh, levels, prec, **kw):
    common = dict(precon="multigrid", solver="fcg", levels=levels, smoother="chebyshev+jacobi",
                  cheby_degree=2, coarse="smooth_jacobi", mgPrecision=prec, tol=1e-8, max_iter=300, **kw)
    return (gpu.Elliptic(mesh, mgGeometry=1, **common), gpu.Elliptic(mesh, mgGeometry=0, **common))


def level_ax_rel(torch, on, off, nlev, dtype, seed):
    rel = []
    for lv in range(nlev):
        n = on.mg_info()[0][lv]["Nlocal"]
        q = torch.from_numpy(np.random.default_rng(seed + lv).uniform(-1, 1, n)).to(dtype).cuda()
        a, b = torch.empty_like(q), torch.empty_like(q)
        on.mg_level(lv, "ax", q, a)
        off.mg_level(lv, "ax", q, b)
        torch.cuda.synchronize()
        rel.append(float(torch.max(torch.abs(a.double() - b.double())) / torch.max(torch.abs(b.double()))))
    return rel


@pytest.mark.parametrize("N", [2, 3, 5, 7, 9])
@pytest.mark.parametrize("prec", [0, 1])
def test_corner_geometry_level_operators(gpu, torch_mod, N, prec):
    torch = torch_mod
    levels = [N] + ([N // 2 + 1] if N > 3 else []) + [1]
    levels = sorted(set(levels), reverse=True)
    mesh = gpu.BoxMesh(4, 3, 3, N, "kershaw", 0.3)
    for kw in ({}, {"lambda0": 1.0, "lambda1": 3.0, "poisson": False}):
        on, off = handles(gpu, mesh, levels, prec, **kw)
        dtype = torch.float64 if prec == 1 else torch.float32
        rel = level_ax_rel(torch, on, off, len(levels), dtype, 10 * N)
        print("N=%d prec=%d %s levels %s rel %s" % (N, prec, "helmholtz" if kw else "poisson", levels, rel),
              flush=True)
        bar = 1e-13 if prec == 1 else 1e-5
        assert max(rel) < bar, rel


@pytest.mark.parametrize("N", [2, 3, 4, 5, 6, 7, 8, 9])
@pytest.mark.parametrize("prec", [0, 1])
def test_corner_variants(gpu, torch_mod, N, prec):
    """Every elements-per-block variant of the corner form, set under its own key, on 63
    elements, most often with a last block that is not full: the bars of the
    level operators (the cofactors of much flatter elements than these cancel
    more: 1.5e-13 in FP64 on a 7x7x1 box).  Order 1 is the coarse level."""
    torch = torch_mod
    mesh = gpu.BoxMesh(7, 3, 3, N, "kershaw", 0.3)
    on, off = handles(gpu, mesh, [N, 1], prec, autotune=0)
    t = "f64" if prec else "f32"
    try:
        for v in (1, 2, 4):
            for n in (N, 1):
                gpu.set_variant("ax", n, t + "_corners", mesh.E, v)
            rel = level_ax_rel(torch, on, off, 2, torch.float64 if prec else torch.float32, N)
            assert all(r < (1e-13 if prec else 1e-5) for r in rel), (v, rel)
    finally:
        for n in (N, 1):
            gpu.set_variant("ax", n, t + "_corners", mesh.E, 0)


@pytest.mark.parametrize("prec", [0, 1])
def test_setup_times_the_corner_form(gpu, torch_mod, prec):
    """A tuned set-up records a variant for the form that each level runs: the corner
    form under its own key where the mesh is trilinear (FP64 above order 7 streams),
    none on a curved mesh, and the entry of the streaming form stays beside it."""
    t = "f64" if prec else "f32"
    orders, E = (9, 5, 1), 5 * 4 * 3
    keys = [("ax", n, t + s, E) for n in orders for s in ("", "_corners")]

    def recorded(mp):
        for k in keys:
            gpu.set_variant(*k, 0)
        el = handles(gpu, gpu.BoxMesh(5, 4, 3, 9, mp, 0.3 if mp == "kershaw" else 0.0), list(orders), prec,
                     autotune=1)[0]
        del el
        got = [gpu.tuned_variant(*k) for k in keys]
        for k in keys:
            gpu.set_variant(*k, 0)
        return got

    got = recorded("kershaw")
    assert all(v in (1, 2, 4) for v in got[::2]), got
    assert all((v == 0) if prec and n == 9 else v in (1, 2, 4) for n, v in zip(orders, got[1::2])), got
    assert not any(recorded("sine")[1::2])


def test_curved_mesh_unchanged(gpu, torch_mod):
    """Sine-mapped nodes are not trilinear: the option has no effect."""
    torch = torch_mod
    mesh = gpu.BoxMesh(3, 3, 2, 5, "sine", 0.0)
    on, off = handles(gpu, mesh, [5, 3, 1], 0)
    rel = level_ax_rel(torch, on, off, 3, torch.float32, 1)
    assert max(rel) == 0.0, rel


@pytest.mark.parametrize("prec", [0, 1])
def test_solves_match(gpu, torch_mod, prec):
    torch = torch_mod
    mesh = gpu.BoxMesh(6, 5, 5, 7, "kershaw", 0.3)
    on, off = handles(gpu, mesh, [7, 3, 1], prec)
    rhs = torch.from_numpy(np.random.default_rng(4).uniform(-1, 1, mesh.Nlocal)).cuda()
    xa, xb = torch.zeros_like(rhs), torch.zeros_like(rhs)
    sa = on.solve(rhs.clone(), xa)
    sb = off.solve(rhs.clone(), xb)
    print("prec %d iterations corner %d stored %d" % (prec, sa["iterations"], sb["iterations"]), flush=True)
    assert sa["converged"] and sb["converged"]
    assert abs(sa["iterations"] - sb["iterations"]) <= 1
    assert float(torch.max(torch.abs(xa - xb)) / torch.max(torch.abs(xb))) < 1e-8


def test_rotated_re2_mesh(gpu, torch_mod, tmp_path):
    """Elements whose corners come in rotated orders (the map's axes differ per element)."""
    import oracle.re2 as r2
    torch = torch_mod
    c = r2.box_corners(3, 3, 2)
    rots = r2.rotations()
    rng = np.random.default_rng(5)
    for e in range(c.shape[0]):
        c[e] = c[e][rots[rng.integers(0, 24)]]
    c[..., 0] += 0.1 * c[..., 1] * c[..., 2]   # a trilinear (not affine) distortion
    path = tmp_path / "rot.re2"
    r2.write(path, c)
    mesh = gpu.Re2Mesh(path, 7)
    on, off = handles(gpu, mesh, [7, 3, 1], 1)
    rel = level_ax_rel(torch, on, off, 3, torch.float64, 2)
    assert max(rel) < 1e-13, rel
