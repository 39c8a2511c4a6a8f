"""The lattice-to-lattice kernel (HOLO_FP32_SPLIT, sources and targets both on
uniform lattices) at the edges of its tiles, forms and detection.

Bar: relative L2 <= 1e-6 against the FP64 oracle, as for every FP32-split path.
Option "grid_pairs" = 0 keeps such calls on the 16-row kernels; calls whose
targets are no lattice give the same bits with the option on and off.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LAM = 632.8e-9


def rel_l2(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def lattice(nx, ny, px, py, x0=0.0, y0=0.0, z=0.0):
    x = x0 + (np.arange(nx) - (nx - 1) / 2.0) * px
    y = y0 + (np.arange(ny) - (ny - 1) / 2.0) * py
    X, Y = np.meshgrid(x, y, indexing="ij")
    return np.stack([X.ravel(), Y.ravel(), np.full(X.size, z)], 1)


def weights(seed, n):
    g = np.random.default_rng(seed)
    return g.random(n), g.random(n) * 2 * np.pi


def both(pkg, f):
    """f() with the option on and off."""
    y1 = f()
    pkg.set_option("grid_pairs", 0)
    y0 = f()
    pkg.set_option("grid_pairs", 1)
    return y1, y0


def check(pkg, ctx, oracle, u, v, sign=1, obliquity=False, seed=0, other=True):
    """Against the oracle, and (other) not the 16-row kernels' bits."""
    amp, phase = weights(seed, len(u))
    plan = ctx.plan(u)
    y1, y0 = both(pkg, lambda: plan.transform(amp, phase, v, sign, LAM, pkg.FP32_SPLIT,
                                              obliquity=obliquity))
    ref = oracle.transform_full(sign, LAM, amp, phase, u, v, obliquity=obliquity)
    print(f"rel L2 {rel_l2(y1, ref):.2e} (16-row kernels {rel_l2(y0, ref):.2e})")
    assert rel_l2(y1, ref) <= 1e-6
    assert np.array_equal(y1, y0) != other


# one tile, a tile less and more by one row or column, wide tiles whose second
# half is missing, and enough tiles for every wave to take a wide one
@pytest.mark.parametrize("src", [(16, 16), (17, 16), (31, 33), (32, 64), (33, 65), (64, 96),
                                 (96, 200)])
@pytest.mark.parametrize("tgt", [(16, 16), (16, 33), (31, 32), (33, 65)])
def test_tile_edges(pkg, ctx, oracle, src, tgt):
    check(pkg, ctx, oracle, lattice(*src, 10e-6, 8e-6), lattice(*tgt, 7e-6, 7.56e-6, z=0.3))


def form(src, sp, tgt, tp, off, z, columns):
    """The kernel's form for centred lattices (sides, pitches), the targets moved
    by off, with source tiles of 32 rows by `columns`, from the bounds of its
    dropped terms restated in FP64: "far", "near" or None."""
    def reach(n, p, m, q, o, tile):
        sides = [abs((n - 1) / 2 * p), (-(-n // tile) * tile - tile / 2) * abs(p)]
        s = (-sides[0] + (tile - 1) / 2 * p, -sides[0] + sides[1] - p / 2)
        t0 = o - (m - 1) / 2 * q
        t = (t0 + 15.5 * q, t0 + (-(-m // 32) * 32 - 16.5) * q)
        r = max(abs(a - b) for a in t for b in s)
        h = 15.5 * q + (tile - 1) / 2 * p
        return 2 * r * h + h * h
    P = reach(src[0], sp[0], tgt[0], tp[0], off[0], 32)
    Q = reach(src[1], sp[1], tgt[1], tp[1], off[1], columns)
    ia, i2 = 1 / (z * LAM), 1 / z ** 2
    cross = np.pi / 2 * ia * i2 * P * Q
    c3 = ia * i2 * i2 / 16
    cubic, sq = 6 * np.pi * c3 * P * Q * (P + Q), (P + Q) * i2
    if cross <= 2.4e-3 and cubic <= 1e-6 and c3 * max(P, Q) ** 3 <= 1e-8 and sq * sq <= 1e-7:
        return "far"
    q4 = 5 / 128 * (P + Q) ** 4 * ia * i2 ** 3
    return "near" if cross <= 0.12 and cubic <= 4e-4 and q4 <= 1e-8 and sq ** 3 <= 1e-7 else None


# from the far form with wide tiles to what only the 16-row kernels take (then
# bit for bit theirs)
@pytest.mark.parametrize("z", [0.35, 0.1, 0.06, 0.045, 0.02])
@pytest.mark.parametrize("sign, obliquity", [(1, False), (-1, True)])
def test_forms(pkg, ctx, oracle, z, sign, obliquity):
    src, sp, tgt, tp, off = (128, 256), (10e-6, 10e-6), (40, 48), (20e-6, 15e-6), (1.5e-3, -1e-3)
    forms = [form(src, sp, tgt, tp, off, z, c) for c in (64, 32)]
    print(f"z {z}: wide {forms[0]}, narrow {forms[1]}")
    check(pkg, ctx, oracle, lattice(*src, *sp), lattice(*tgt, *tp, *off, z), sign, obliquity,
          other=any(forms))


@pytest.mark.parametrize("flips", [(-1, 1, 1, 1), (1, -1, 1, -1), (-1, -1, -1, -1)])
def test_descending_pitches_and_planes(pkg, ctx, oracle, flips):
    """Any order of rows and columns, sources above the targets."""
    a, b, c, d = flips
    check(pkg, ctx, oracle, lattice(48, 80, a * 9e-6, b * 7e-6, z=0.3),
          lattice(35, 50, c * 6e-6, d * 8e-6, 1e-3, 0, 0.0), -1)


@pytest.mark.parametrize("splits", [0, 1, 3, 7])
def test_generator_planes(pkg, ctx, oracle, workloads, splits):
    """Planes of the reference's generator on both sides: copies of point 0 after
    the lattice (summed once as sources, repeated as targets)."""
    u = workloads.reference_plane(9029, 1e-3, 0.0, 1.0, (1e-4, -2e-4))
    v = workloads.reference_plane(2029, 5e-4, 0.3, 0.8)
    pkg.set_option("splits", splits)
    check(pkg, ctx, oracle, u, v)
    pkg.set_option("splits", 0)


def test_tail_of_arbitrary_sources(pkg, ctx, oracle):
    g = np.random.default_rng(5)
    tail = np.zeros((40, 3))
    tail[:, :2] = (g.random((40, 2)) - 0.5) * 2e-3
    u = np.concatenate([lattice(64, 96, 10e-6, 10e-6), tail])
    check(pkg, ctx, oracle, u, lattice(40, 40, 8e-6, 8e-6, z=0.25))


def _moved(v, i, d, by):
    w = v.copy()
    w[i, d] += by
    return w


def test_targets_off_a_lattice_keep_their_path(pkg, ctx, oracle):
    """One target off its place, short or permuted lattices, several planes: the
    16-row kernels' bits."""
    u = lattice(64, 64, 10e-6, 10e-6)
    v = lattice(40, 36, 8e-6, 8e-6, z=0.3)
    g = np.random.default_rng(3)
    x = g.random(40) * 1e-3
    X, Y = np.meshgrid(np.sort(x), np.arange(36) * 8e-6, indexing="ij")
    others = [_moved(v, 700, 0, 1e-9), _moved(v, len(v) - 1, 1, 1e-9), _moved(v, 5, 2, 1e-9),
              v[g.permutation(len(v))], v[:-1], v[:300],
              v.reshape(40, 36, 3).transpose(1, 0, 2).reshape(-1, 3),
              np.concatenate([v, v[1:2]]), lattice(15, 64, 8e-6, 8e-6, z=0.3),
              lattice(64, 15, 8e-6, 8e-6, z=0.3),
              np.stack([X.ravel(), Y.ravel(), np.full(X.size, 0.3)], 1),
              lattice(40, 36, 0.0, 8e-6, z=0.3), lattice(40, 36, 8e-6, 8e-6, z=0.0)[:0]]
    for w in others:
        if len(w):
            check(pkg, ctx, oracle, u, np.ascontiguousarray(w), other=False)


@pytest.mark.parametrize("z", [0.3, 0.08])
@pytest.mark.parametrize("scale", [1e-30, 1.0, 1e25])
def test_complex_weights_scales_and_adjoint(pkg, ctx, oracle, z, scale):
    """Complex weights and the adjoint (both lattices change places), weights of
    any scale, a row of tiles far below or zero beside the others."""
    u, v = lattice(50, 70, 10e-6, 9e-6), lattice(33, 44, 8e-6, 8e-6, 5e-4, 0, z)
    g = np.random.default_rng(int(z * 100))
    w = (g.standard_normal(len(u)) + 1j * g.standard_normal(len(u))) * scale
    w.reshape(50, 70)[32:40] *= 1e-6
    w.reshape(50, 70)[40:] = 0.0
    y1, y0 = both(pkg, lambda: ctx.plan(u).transform_complex(w, v, -1, LAM, pkg.FP32_SPLIT))
    ref = oracle.transform_cartesian(-1, LAM, w / scale, u, v)
    assert rel_l2(y1 / scale, ref) <= 1e-6 and not np.array_equal(y1, y0)
    amp, theta = weights(7, len(u))
    gz = g.standard_normal(len(v)) + 1j * g.standard_normal(len(v))
    ga, gt = ctx.plan(v).adjoint(gz, amp, theta, u, +1, LAM, pkg.FP32_SPLIT)
    ra, rt = oracle.adjoint(+1, LAM, amp, theta, u, gz, v)
    assert rel_l2(ga, ra) <= 1e-6 and rel_l2(gt, rt) <= 1e-6


@pytest.mark.parametrize("seed", range(12))
def test_random_lattices(pkg, ctx, seed):
    """Seeded pairs of lattices: sides, pitches, offsets, 3 cm to 1 m, 400 - 700
    nm, either sign, with or without obliquity, within 1e-6 of FP64."""
    g = np.random.default_rng(300 + seed)
    sides = [int(s) for s in g.integers(16, 150, 4)]
    pitch = g.uniform(2e-6, 20e-6, 4) * g.choice([-1, 1], 4)
    off = g.uniform(-3e-3, 3e-3, 4)
    z = float(np.exp(g.uniform(np.log(0.03), 0.0)))
    u = lattice(sides[0], sides[1], pitch[0], pitch[1], off[0], off[1], 0.01)
    v = lattice(sides[2], sides[3], pitch[2], pitch[3], off[2], off[3], 0.01 + z)
    lam, sign, obl = g.uniform(400e-9, 700e-9), int(g.choice([-1, 1])), bool(g.random() < 0.3)
    amp, phase = weights(seed, len(u))
    plan = ctx.plan(u)
    ref = plan.transform(amp, phase, v, sign, lam, pkg.FP64, obliquity=obl)
    y1, y0 = both(pkg, lambda: plan.transform(amp, phase, v, sign, lam, pkg.FP32_SPLIT,
                                              obliquity=obl))
    print(f"z {z:.3f}: rel L2 {rel_l2(y1, ref):.2e} (16-row kernels {rel_l2(y0, ref):.2e})")
    assert rel_l2(y1, ref) <= 1e-6


def test_graph_replays(pkg, ctx):
    """Captured into a HIP graph and replayed on changed weights and targets (a
    lattice, then none), with eager work between the replays."""
    import torch
    dev = torch.device("cuda")
    u = torch.from_numpy(lattice(64, 64, 10e-6, 10e-6)).to(dev)
    v1 = torch.from_numpy(lattice(40, 48, 8e-6, 8e-6, z=0.3)).to(dev)
    v2 = v1.clone()
    v2[100, 0] += 1e-9
    plan = ctx.plan(u)
    g = torch.Generator(device=dev).manual_seed(1)
    ws = [torch.rand((2, 4096), dtype=torch.float64, device=dev, generator=g) for _ in range(3)]
    a, p, v = torch.empty_like(ws[0][0]), torch.empty_like(ws[0][0]), v1.clone()
    call = lambda: plan.transform(a, p, v, 1, LAM, pkg.FP32_SPLIT)
    a.copy_(ws[0][0])
    p.copy_(ws[0][1])
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        y = call()
    for k, vk in ((1, v1), (2, v2), (0, v1), (1, v2)):
        a.copy_(ws[k][0])
        p.copy_(ws[k][1])
        v.copy_(vk)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, call())
