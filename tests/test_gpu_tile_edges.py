"""GPU: kernels whose tiling depends on the grid, at the sizes where a tile can go wrong."""
from __future__ import annotations

import numpy as np
import pytest

from tests._helpers import from_dev, random_state, to_dev

pytestmark = pytest.mark.gpu

OPT = (2, False, False, 0, False, False, 1)


def _case(nx, ny, nz, passive, seed=3):
    from lex_amd import _lib
    gr, phys, base = random_state(nx, ny, nz, seed=seed, passive=passive, vel=2.0)
    g = _lib.grid(nx, ny, nz, gr.dx, gr.dy, gr.dz)
    return g, tuple(to_dev(a) for a in phys), tuple(to_dev(a) for a in base[:5])


# marches of 1, 2, 5, 9 and 16 cells with full and partial last tiles, ny mod 4 of 0..3,
# one, two and three waves per column; substeps in pairs and (the last three) one by one
@pytest.mark.parametrize("shape,passive", [((8, 9, 16), 0), ((40, 41, 40), 0), ((67, 62, 64), 2), ((97, 91, 70), 1),
                                           ((157, 160, 130), 2), ((203, 199, 9), 0), ((201, 202, 50), 1),
                                           ((30, 23, 150), 0)], ids=str)
def test_stage_tiles_equal_per_operator_kernels(shape, passive):
    """One step with the stage kernel against one kernel per reference routine: the same
    arithmetic up to operation order, a few FP32 ulps of each field (64, as for the other
    fused kernels)."""
    from lex_amd import one_sprint_functions as sp
    g, phys, base = _case(*shape, passive)
    got = sp.fused_step(tuple(a.clone() for a in phys), base, g, OPT, dt=0.2, n_sound=4)
    ref = sp.fused_step(tuple(a.clone() for a in phys), base, g, OPT, dt=0.2, n_sound=4, impl=1)
    for q, (a, b) in enumerate(zip(got, ref)):
        a, b = from_dev(a), from_dev(b)
        assert np.isfinite(b).all()
        ulp = float(np.spacing(np.float32(np.abs(b).max())))
        assert np.max(np.abs(a - b)) <= 64 * ulp, (q, np.max(np.abs(a - b)) / ulp)


# one and two levels per lane, columns of one wave and of several with one level left over,
# even and odd nz, marches of one and of several cells; a thread per cell above 128 levels
@pytest.mark.parametrize("shape", [(8, 9, 24), (17, 9, 64), (9, 7, 65), (33, 18, 128), (6, 6, 129), (20, 21, 200),
                                   (161, 120, 73), (9, 10, 192), (12, 6, 193), (90, 91, 250), (7, 8, 321)], ids=str)
def test_acoustic_substep_against_oracle(shape):
    """One substep against the FP64 oracle, the input's ghosts not periodic images (an initial
    state's need not be); error within 8x the FP32 oracle's own, as for the other operators."""
    import torch
    from lex_amd import _lib
    from oracle import lex_oracle as o
    from tests._helpers import check_fp32
    nx, ny, nz = shape
    gr, phys, base = random_state(nx, ny, nz, seed=5, vel=2.0)
    rng = np.random.default_rng(7)
    th, u, v, w, p = phys[:5]
    p = np.asarray(p + rng.normal(0, 1e-5, p.shape), np.float32)
    ps = np.asarray(p + rng.normal(0, 1e-6, p.shape), np.float32)
    u, v, w, th = (np.asarray(a, np.float32) for a in (u, v, w, th))
    ru, rv, rw = (np.asarray(rng.normal(0, 1e-2, s), np.float32)
                  for s in ((nx + 1, ny, nz), (nx, ny + 1, nz), (nx, ny, nz + 1)))
    rho, pi0 = (np.asarray(base[q], np.float32) for q in (1, 3))
    ref = []
    for dt in (np.float64, np.float32):
        f = lambda a: np.asarray(a, dt)  # noqa: E731
        ref.append(o.sound_rk_step(f(u), f(v), f(w), f(pi0), f(p), f(ps), f(ru), f(rv), f(rw), f(th), f(rho), 1, 0.1, gr))
    ins = [to_dev(a) for a in (rho[3, 3], pi0[3, 3], u, v, w, p, ps, ru, rv, rw, th)]
    out = [torch.full_like(t, float("nan")) for t in ins[2:6]]
    g = _lib.grid(nx, ny, nz, gr.dx, gr.dy, gr.dz)
    _lib.call("lex_acoustic_substep", g, *[_lib.ptr(t) for t in ins], 0.1, *[_lib.ptr(t) for t in out], _lib.stream())
    for name, got, r64, r32 in zip("u v w p".split(), out, *ref):
        check_fp32(from_dev(got), r64, r32, name)


# an infinity in the middle of a lane's levels, at the last level of a wave and above the floor
@pytest.mark.parametrize("shape,levels", [((9, 10, 24), (1, 12)), ((9, 10, 70), (5, 63, 64)),
                                          ((9, 10, 140), (127, 128)), ((9, 10, 230), (127, 128))], ids=str)
def test_acoustic_substep_of_a_blown_up_state(shape, levels):
    """Infinite w and u: the kernels give the infinities and NaNs of the oracle's IEEE arithmetic,
    one substep at a time and two in one launch."""
    import torch
    from lex_amd import _lib
    from oracle import lex_oracle as o
    nx, ny, nz = shape
    gr, phys, base = random_state(nx, ny, nz, seed=5, vel=2.0)
    rng = np.random.default_rng(7)
    th, u, v, w, p = (np.array(a, np.float32) for a in phys[:5])
    ps = np.asarray(p + rng.normal(0, 1e-6, p.shape), np.float32)
    for n, k in enumerate(levels):
        w[6 - n, 6 + n, k + 1] = np.inf if n % 2 == 0 else -np.inf
        u[7, 4, k + 1] = -np.inf
    ru, rv, rw = (np.asarray(rng.normal(0, 1e-2, s), np.float32)
                  for s in ((nx + 1, ny, nz), (nx, ny + 1, nz), (nx, ny, nz + 1)))
    rho, pi0 = (np.asarray(base[q], np.float32) for q in (1, 3))
    fixed = [to_dev(a) for a in (ps, ru, rv, rw, th)]
    cols = [to_dev(a) for a in (rho[3, 3], pi0[3, 3])]
    g = _lib.grid(nx, ny, nz, gr.dx, gr.dy, gr.dz)
    f = lambda a: np.asarray(a, np.float64)  # noqa: E731

    def call(name, state):
        out = [torch.zeros_like(t) for t in state]
        _lib.call(name, g, *[_lib.ptr(t) for t in (*cols, *state, *fixed)], 0.1, *[_lib.ptr(t) for t in out],
                  _lib.stream())
        return out

    start = [to_dev(a) for a in (u, v, w, p)]
    one = call("lex_acoustic_substep", start)
    for n, got in ((1, one), (2, call("lex_acoustic_substep", one)), (2, call("lex_acoustic_substep_pair", start))):
        with np.errstate(invalid="ignore"):
            ref = o.sound_rk_step(f(u), f(v), f(w), f(pi0), f(p), f(ps), f(ru), f(rv), f(rw), f(th), f(rho), n, 0.1, gr)
        for name, a, b in zip("u v w p".split(), got, ref):
            a = from_dev(a)
            assert np.array_equal(np.isnan(a), np.isnan(b)), (name, n)
            assert np.array_equal(a[np.isinf(b)], b[np.isinf(b)]) and np.isinf(b).sum() == np.isinf(a).sum(), (name, n)
    assert torch.isinf(one[3]).any()


# one and two levels per lane, columns of one wave and of two, full and partial strips of
# rows, marches of one and of several cells, the last one shorter; one and several rounds of
# workgroups, more strips than a round has; more cells in x than a launch's second and third dimension
@pytest.mark.parametrize("shape", [(6, 6, 24), (7, 13, 64), (100, 13, 40), (17, 9, 65), (33, 21, 128), (9, 7, 129),
                                   (20, 9, 256), (181, 147, 71), (300, 60, 33), (23, 3200, 6), (19, 1310, 65),
                                   (40, 530, 130), (401, 127, 129), (251, 203, 192), (65543, 6, 129), (132009, 6, 9)], ids=str)
def test_acoustic_pair_is_two_substeps(shape):
    """Two substeps in one launch equal two launches bit for bit; the input's ghosts are not
    periodic images."""
    import torch
    from lex_amd import _lib
    nx, ny, nz = shape
    gen = torch.Generator(device="cuda").manual_seed(3)
    R = lambda s, *n: s * torch.randn(*n, generator=gen, device="cuda")  # noqa: E731
    u, v = R(2.0, nx + 7, ny + 6, nz + 2), R(2.0, nx + 6, ny + 7, nz + 2)
    w, p = R(2.0, nx + 6, ny + 6, nz + 3), R(1e-5, nx + 6, ny + 6, nz + 2)
    tr, ps = 300.0 + R(1.0, nx + 6, ny + 6, nz + 2), p + R(1e-6, nx + 6, ny + 6, nz + 2)
    ru, rv, rw = R(1e-2, nx + 1, ny, nz), R(1e-2, nx, ny + 1, nz), R(1e-2, nx, ny, nz + 1)
    rho, pi0 = 1.0 + 0.1 * R(1.0, nz + 2).abs(), 0.9 + R(1e-2, nz + 2)
    g = _lib.grid(nx, ny, nz, 100.0, 110.0, 90.0)

    def call(name, state):
        out = [torch.full_like(t, float("nan")) for t in state]
        ins = (rho, pi0, *state, ps, ru, rv, rw, tr)
        _lib.call(name, g, *[_lib.ptr(t) for t in ins], 0.1, *[_lib.ptr(t) for t in out], _lib.stream())
        return out

    want = call("lex_acoustic_substep", call("lex_acoustic_substep", (u, v, w, p)))
    for name, a, b in zip("u v w p".split(), call("lex_acoustic_substep_pair", (u, v, w, p)), want):
        assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(), b.nan_to_num()), name


# marches of 2, 4 and 5 cells, the last one shorter
@pytest.mark.parametrize("shape", [(101, 90, 24), (110, 130, 64), (97, 91, 70)], ids=str)
def test_smagorinsky_marches_equal_routine_chain(shape):
    from tests.test_gpu_step import test_fused_smagorinsky_equals_routine_chain as chain
    chain(shape, 1)


# one and two levels per lane, the smallest and the fullest columns of each, one level left
# over, marches of one and of several cells; above 128 levels the workgroup-per-column form with
# three and four waves, partly filled and full
@pytest.mark.parametrize("shape", [(8, 9, 6), (17, 9, 64), (9, 7, 65), (9, 8, 127), (12, 11, 128), (161, 160, 33),
                                   (8, 9, 129), (7, 10, 192), (6, 7, 193), (9, 8, 256)], ids=str)
def test_implicit_substep_against_oracle(shape):
    """One vertically implicit substep against the FP64 oracle (a Thomas solve there); error
    within 8x the FP32 oracle's own, as for the other operators."""
    import torch
    from lex_amd import _lib
    from oracle import lex_oracle as o
    from tests._helpers import check_fp32
    nx, ny, nz = shape
    gr, phys, base = random_state(nx, ny, nz, seed=5, vel=2.0)
    rng = np.random.default_rng(7)
    th, u, v, w, p = (np.asarray(a, np.float32) for a in phys[:5])
    ps = np.asarray(p + rng.normal(0, 1e-6, p.shape), np.float32)
    ru, rv, rw = (np.asarray(rng.normal(0, 1e-2, s), np.float32)
                  for s in ((nx + 1, ny, nz), (nx, ny + 1, nz), (nx, ny, nz + 1)))
    rho, pi0 = (np.asarray(base[q], np.float32) for q in (1, 3))
    ref = []
    for dt in (np.float64, np.float32):
        f = lambda a: np.asarray(a, dt)  # noqa: E731
        ref.append(o.sound_implicit_rk_step(f(u), f(v), f(w), f(pi0), f(p), f(ps), f(ru), f(rv), f(rw), f(th), f(rho),
                                            1, 0.2, gr))
    ins = [to_dev(a) for a in (rho[3, 3], pi0[3, 3], u, v, w, p, ps, ru, rv, rw, th)]
    out = [torch.full_like(t, float("nan")) for t in ins[2:6]]
    g = _lib.grid(nx, ny, nz, gr.dx, gr.dy, gr.dz)
    _lib.call("lex_acoustic_substep_implicit", g, *[_lib.ptr(t) for t in ins], 0.2, 0.6, *[_lib.ptr(t) for t in out],
              _lib.stream())
    for name, got, a0, r64, r32 in zip("u v w p".split(), out, (u, v, w, p), *ref):
        check_fp32(from_dev(got) - a0, r64 - a0, r32 - a0, name)


# one block, several with a last one partly filled, exactly two cells per thread, and the
# loop past the two cells a thread requests ahead (more than 1024 blocks of 512 cells)
@pytest.mark.parametrize("shape", [(6, 6, 6), (19, 23, 17), (32, 32, 64), (96, 96, 60)], ids=str)
def test_bicgstab_first_iterations_against_oracle(shape):
    """Four BiCGSTAB iterations against the FP64 oracle.  The first iterations do not yet
    amplify rounding: the FP32 oracle is 1e-7 to 1e-6 off after them, and the bound is 8x its
    error, as for the other operators."""
    import torch
    from lex_amd import _lib
    from oracle import lex_oracle as o
    from tests._helpers import check_fp32
    nx, ny, nz = shape
    gr = o.Grid(nx, ny, nz, 600.0, 600.0, 300.0)
    rng = np.random.default_rng(11)
    rtt = np.asarray(rng.uniform(200.0, 350.0, gr.shape_c), np.float32)
    rtt[:, :, 0] = rtt[:, :, -1] = 0.0   # no buoyancy: the operator is linear
    b = np.asarray(o.laplace_of_pressure(rtt.astype(np.float64), rng.normal(0, 1e-3, shape), gr), np.float32)
    x0 = np.asarray(rng.normal(0, 1e-4, shape), np.float32)
    ref = [o.bicgstab(lambda x, dt=dt: o.laplace_of_pressure(rtt.astype(dt), x, gr), b.astype(dt), x0.astype(dt), 1e-12,
                      0.0, 4) for dt in (np.float64, np.float32)]
    g = _lib.grid(nx, ny, nz, gr.dx, gr.dy, gr.dz)
    ws = torch.empty(_lib.load().lex_bicgstab_workspace_bytes(g), dtype=torch.uint8, device="cuda")
    rt, bd, xd = to_dev(rtt), to_dev(b), to_dev(x0)
    x = torch.empty_like(xd)
    import ctypes
    k = ctypes.c_int(-99)
    _lib.call("lex_bicgstab", g, _lib.ptr(rt), _lib.ptr(bd), _lib.ptr(xd), _lib.ptr(x), 1e-12, 0.0, 4, _lib.ptr(ws),
              ws.numel(), ctypes.byref(k), _lib.stream())
    assert k.value == ref[0][1] == 4
    check_fp32(from_dev(x), ref[0][0], ref[1][0], "x")


# runs shorter than a step, of one step, and long enough to go round the ring of planes; one
# and several rows and z tiles with and without a remainder; periods of two and three cells,
# which a step's planes and rows run round more than once; 16 and 32 channels either side
@pytest.mark.parametrize("circular", [False, True])
@pytest.mark.parametrize("cin,cout", [(5, 32), (32, 32), (32, 5), (16, 16)])
@pytest.mark.parametrize("shape", [(4, 4, 16), (7, 5, 17), (46, 9, 35), (97, 66, 33), (2, 3, 18), (3, 2, 16),
                                   (2, 2, 3), (2, 21, 40), (19, 3, 40)], ids=str)
def test_convolution_march(shape, cin, cout, circular):
    """One convolution against torch conv3d in float64 on the same BF16 operands: FP32 sums of
    27 cin products, 1e-5 as for the other sizes; the BF16 output is its rounding (2^-8)."""
    import torch
    from lex_amd import sgs_net as sn
    gen = torch.Generator().manual_seed(cin + cout)
    x = torch.randn(*shape, cin, generator=gen)
    W = torch.randn(27, cin, cout, generator=gen) / np.sqrt(27 * cin)
    b = 0.1 * torch.randn(cout, generator=gen)
    xb = x.bfloat16().double().permute(3, 0, 1, 2)[None]
    wb = W.bfloat16().double().view(3, 3, 3, cin, cout).permute(4, 3, 0, 1, 2)
    if circular:
        xb = torch.nn.functional.pad(torch.nn.functional.pad(xb, (0, 0, 1, 1, 1, 1), mode="circular"), (1, 1))
    else:
        xb = torch.nn.functional.pad(xb, (1,) * 6)
    ref = torch.nn.functional.conv3d(xb, wb, b.double())[0].permute(1, 2, 3, 0)
    xd = sn.to_bf16_channels_last(x.cuda())
    yf, _ = sn.conv3d_fwd(xd, shape, W.cuda(), b.cuda(), gelu=False, out_fp32=True, circular=circular)
    yb, pre = sn.conv3d_fwd(xd, shape, W.cuda(), b.cuda(), gelu=False, out_fp32=False, want_pre=True, circular=circular)
    rel = lambda a: float((a.cpu().double().view(*shape, -1)[..., :cout] - ref).norm() / ref.norm())  # noqa: E731
    assert rel(yf) < 1e-5 and rel(pre) < 1e-5 and rel(yb) < 2.0 ** -8


# less than a tile, one tile over and under in each direction, several tiles per workgroup
@pytest.mark.parametrize("cin,cout", [(16, 16), (9, 32), (32, 11), (32, 32)])
@pytest.mark.parametrize("shape", [(5, 6, 7), (9, 4, 16), (4, 9, 33), (50, 47, 18)], ids=str)
def test_conv_weight_gradient(shape, cin, cout):
    """Weight and bias gradient against FP64 sums of the same BF16 operands: FP32 sums of n
    products, whose rounding grows like sqrt(n) of an ulp."""
    import torch
    from lex_amd import sgs_net as sn
    nx, ny, nz = shape
    n, cip, cop = nx * ny * nz, 16 * ((cin + 15) // 16), 16 * ((cout + 15) // 16)
    gen = torch.Generator(device="cuda").manual_seed(2)
    x = torch.randn(n, cip, device="cuda", generator=gen).to(torch.bfloat16)
    gp = torch.randn(n, cop, device="cuda", generator=gen).to(torch.bfloat16)
    dw, db = sn.conv3d_bwd_weight(x, gp, shape, cin, cout)
    xp = torch.zeros(nx + 2, ny + 2, nz + 2, cin, dtype=torch.float64, device="cuda")
    xp[1:-1, 1:-1, 1:-1] = x[:, :cin].double().view(nx, ny, nz, cin)
    g64 = gp[:, :cout].double()
    ref = torch.stack([xp[a:a + nx, b:b + ny, c:c + nz].reshape(n, cin).t() @ g64
                       for a in range(3) for b in range(3) for c in range(3)])
    tol = n ** 0.5 * 2.0 ** -24
    assert float((dw.double() - ref).norm() / ref.norm()) <= tol
    assert float((db.double() - g64.sum(0)).norm() / g64.sum(0).norm()) <= 4 * tol   # sums that cancel


def test_conv_of_an_unaligned_view():
    """An input that starts two bytes off a 16-byte boundary gives the aligned input's bits."""
    import torch
    from lex_amd import _lib
    nx, ny, nz, c = 9, 7, 18, 32
    n = nx * ny * nz
    gen = torch.Generator(device="cuda").manual_seed(4)
    x = torch.randn(n * c, device="cuda", generator=gen).to(torch.bfloat16)
    off = torch.empty(n * c + 1, dtype=torch.bfloat16, device="cuda")[1:].copy_(x)
    assert off.data_ptr() % 16 == 2
    w, b = torch.randn(27, c, c, device="cuda", generator=gen), torch.zeros(c, device="cuda")
    wp = torch.empty(c * 27 * c, dtype=torch.bfloat16, device="cuda")
    _lib.call("lex_conv3d_pack_weights", _lib.ptr(w), c, c, 0, _lib.ptr(wp), _lib.stream())
    out = [torch.zeros(n, c, dtype=torch.bfloat16, device="cuda") for _ in range(2)]
    for t, y in zip((x, off), out):
        _lib.call("lex_conv3d_bf16_fwd", nx, ny, nz, c, c, _lib.ptr(t), _lib.ptr(wp), _lib.ptr(b), 1, 0, _lib.ptr(y),
                  None, None, _lib.stream())
    assert torch.equal(*out)


@pytest.mark.parametrize("cin,cout", [(16, 32), (32, 32), (32, 16), (16, 5)])
def test_conv_with_unaligned_outputs(cin, cout):
    """Outputs, pre-activations and the pre-activations that the data gradient reads, one element
    off a 16-byte boundary: the bits of aligned buffers, and nothing beside them."""
    import torch
    from lex_amd import _lib
    nx, ny, nz = 6, 7, 18
    n, cop = nx * ny * nz, 16 * ((cout + 15) // 16)
    gen = torch.Generator(device="cuda").manual_seed(4)
    x = torch.randn(n * cin, device="cuda", generator=gen).to(torch.bfloat16)
    w, b = torch.randn(27, cin, cout, device="cuda", generator=gen), torch.randn(cop, device="cuda", generator=gen)
    wp = torch.empty(cop * 28 * cin, dtype=torch.bfloat16, device="cuda")
    _lib.call("lex_conv3d_pack_weights", _lib.ptr(w), cin, cout, 0, _lib.ptr(wp), _lib.stream())

    def buf(count, dtype, off, fill=-7.0):
        t = torch.full((count + off + 8,), fill, dtype=dtype, device="cuda")
        assert t.data_ptr() % 16 == 0
        return t, t[off:off + count]

    def run(off):
        whole, out = [], []
        for c, dt in ((cop, torch.bfloat16), (cop, torch.float32), (cout, torch.float32)):
            t, v = buf(n * c, dt, off)
            whole.append(t)
            out.append(v)
        y, pre, yf = (_lib.ptr(v) for v in out)
        args = (nx, ny, nz, cin, cout, _lib.ptr(x), _lib.ptr(wp), _lib.ptr(b))
        _lib.call("lex_conv3d_bf16_fwd", *args, 1, 0, y, None, pre, _lib.stream())
        _lib.call("lex_conv3d_bf16_fwd", *args, 1, 1, None, yf, None, _lib.stream())
        if cop == 32:   # the same products as a data gradient, times the GELU's derivative at pre
            t, v = buf(n * cop, torch.bfloat16, off)
            whole.append(t)
            out.append(v)
            _lib.call("lex_conv3d_bf16_bwd_data_gelu", nx, ny, nz, cout, cin, _lib.ptr(x), _lib.ptr(wp), _lib.ptr(b),
                      pre, _lib.ptr(v), _lib.stream())
        for t, v in zip(whole, out):
            assert bool((t[:off] == -7.0).all()) and bool((t[off + v.numel():] == -7.0).all())
        return out

    for a, c in zip(run(0), run(1)):
        assert c.data_ptr() % 16 in (2, 4) and torch.equal(a, c)


@pytest.mark.parametrize("cin,cout,circular", [(16, 16, False), (16, 32, True), (32, 16, True), (32, 32, False)])
def test_conv_of_an_unaligned_view_takes_no_memory(cin, cout, circular):
    """An input off a 16-byte boundary, whole and partial tiles, all outputs: the aligned input's
    bits, and the device's free memory as before (the calls may run where none can be taken)."""
    import torch
    from lex_amd import _lib
    nx, ny, nz = 70, 67, 275
    n = nx * ny * nz
    gen = torch.Generator(device="cuda").manual_seed(4)
    buf = torch.empty(n * cin + 8, dtype=torch.bfloat16, device="cuda")
    x = torch.randn(n * cin, device="cuda", generator=gen).to(torch.bfloat16)
    w, b = torch.randn(27, cin, cout, device="cuda", generator=gen), torch.randn(cout, device="cuda", generator=gen)
    wp = torch.empty(cout * 28 * cin, dtype=torch.bfloat16, device="cuda")
    _lib.call("lex_conv3d_pack_weights", _lib.ptr(w), cin, cout, 0, _lib.ptr(wp), _lib.stream())
    entry = "lex_conv3d_bf16_fwd_circular" if circular else "lex_conv3d_bf16_fwd"

    def outputs():
        return [torch.full((n * cout,), -7.0, dtype=t, device="cuda")
                for t in (torch.bfloat16, torch.float32, torch.float32, torch.bfloat16)]

    def run(v, out):
        y, pre, yf, dx = (_lib.ptr(t) for t in out)
        args = (nx, ny, nz, cin, cout, _lib.ptr(v), _lib.ptr(wp), _lib.ptr(b))
        _lib.call(entry, *args, 1, 0, y, None, pre, _lib.stream())
        _lib.call(entry, *args, 0, 1, None, yf, None, _lib.stream())
        if cout == 32:
            _lib.call("lex_conv3d_bf16_bwd_data_gelu", nx, ny, nz, cout, cin, *args[5:], pre, dx, _lib.stream())
        torch.cuda.synchronize()

    want, got = outputs(), outputs()
    run(x, want)
    for off in (1, 4):
        v = buf[off:off + n * cin].copy_(x)
        assert v.data_ptr() % 16 == 2 * off
        free = torch.cuda.mem_get_info()[0]
        run(v, got)
        assert free - torch.cuda.mem_get_info()[0] < n * cin   # half of x
        for a, c in zip(got, want):
            assert torch.equal(a, c)
            a.fill_(-7.0)


@pytest.mark.parametrize("cin,cout", [(5, 32), (16, 16), (16, 32), (32, 32), (32, 5)])
def test_conv_of_an_infinite_cell(cin, cout):
    """An infinite activation gives an infinity of the weight's sign at each of the 27 outputs that
    it reaches, and leaves the others as they are."""
    import torch
    from lex_amd import sgs_net as sn
    shape = (9, 10, 35)
    gen = torch.Generator().manual_seed(3)
    x = torch.randn(*shape, cin, generator=gen)
    w, b = torch.randn(27, cin, cout, generator=gen), torch.randn(cout, generator=gen)
    run = lambda t: sn.conv3d_fwd(sn.to_bf16_channels_last(t.cuda()), shape, w.cuda(), b.cuda(), gelu=False,  # noqa: E731
                                  out_fp32=True)[0].cpu().view(*shape, cout)
    want = run(x)
    for cell, c, v in (((4, 5, 17), 0, float("inf")), ((1, 7, 30), cin - 1, -float("inf"))):
        x[(*cell, c)] = v
        for tap in range(27):
            o = [a - d + 1 for a, d in zip(cell, (tap // 9, tap // 3 % 3, tap % 3))]
            want[tuple(o)] = v * w[tap, c].sign()
    assert torch.equal(run(x), want)


@pytest.mark.parametrize("shape", [(1, 262153, 1), (262153, 2, 2), (2, 1, 1048601)], ids=str)
def test_conv_of_a_long_grid(shape):
    """More rows than a launch has in its second dimension, and as long in x and z."""
    import torch
    from lex_amd import sgs_net as sn
    gen = torch.Generator().manual_seed(3)
    x, w = torch.randn(*shape, 5, generator=gen), torch.randn(27, 5, 5, generator=gen)
    xb, wb = x.bfloat16().double().permute(3, 0, 1, 2)[None], w.bfloat16().double().view(3, 3, 3, 5, 5)
    ref = torch.nn.functional.conv3d(xb, wb.permute(4, 3, 0, 1, 2), padding=1)[0].permute(1, 2, 3, 0)
    got, _ = sn.conv3d_fwd(sn.to_bf16_channels_last(x.cuda()), shape, w.cuda(), torch.zeros(5, device="cuda"),
                           gelu=False, out_fp32=True)
    assert float((got.cpu().double().view(*shape, 5) - ref).norm() / ref.norm()) < 1e-5
