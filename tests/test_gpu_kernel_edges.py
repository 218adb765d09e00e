"""Kernels at the sizes where their tiling can go wrong: block edges,
remainders, the smallest grids and both sides of each dispatch rule."""
import ctypes as C
import os
import subprocess
import sys
import time

import numpy as np
import pytest

import chybrid
import orc
from gpu_cases import (as_particles, context, grid_of, opts, oracle_sorted, push_params_of, random_particles, relmax, upload,
                       vlasov_from)

pytestmark = pytest.mark.gpu


def _moments(g, rng, amp=0.2):
    n = 1 + amp * rng.uniform(-1, 1, g.nc)
    return [n] + [0.1 * rng.standard_normal(g.nc) for _ in range(3)]


# one block of columns is 256, a group of planes 4; the 128-plane grid is the
# largest of the FP64 column stencil, the 129-plane one goes to the tiles
@pytest.mark.parametrize("extra", ["", "-B0x 1e-5 -B0y 2e-5", "--lhs-type laplacian"])
@pytest.mark.parametrize("N", [(3, 3, 3), (16, 16, 4), (17, 15, 9), (257, 3, 7), (40, 24, 33), (128, 128, 128),
                               (128, 128, 129)])
def test_stencil_is_the_oracles_bit_for_bit(N, extra):
    rng = np.random.default_rng(11)
    with context(opts(N, extra=extra)) as ctx:
        g = grid_of(ctx.prm)
        mom = _moments(g, rng)
        ctx.set_moments(vlasov_from(mom))
        x = rng.standard_normal(g.nc)
        y = ctx.lhs_apply(x)
        yt = ctx.lhs_apply(x, transpose=True)
        K, lt = list(ctx.prm.kappa_e), ctx.prm.lhs_type
    assert np.array_equal(y, orc.lhs_apply(g, K, mom[0], x, lhs_type=lt))
    ref = orc.lhs_apply(g, K, mom[0], x, lhs_type=lt, transpose=True)
    # the oracle scatters its rows: the same 19 products a node, in another order
    assert np.abs(yt - ref).max() <= 19 * 2.0 ** -52 * np.abs(ref).max() * 19


# the one-workgroup 2-D correction: planes of 16 to 2048 nodes with even and
# odd log2 lengths and the longest lines it takes, every pair of 16, 32 and 64
# points in registers up to that size; beyond it the separate
# launches, at one and several rows a block, and with x lines whose inverse
# (2048 points in FP64) is a launch of its own.  The symbol of the FFT stage is a
# sum that cancels towards the weakest mode: lambda_min / A0 = (1 - cos(2 pi /
# N)) / (2 + 1 + Kz^2), and its 8 roundings on each side, in another order,
# bound the agreement with the oracle.
@pytest.mark.parametrize("prec,base", [("fp64", 1e-12), ("mixed", 2e-5)])
@pytest.mark.parametrize("N", [(4, 4, 4), (8, 4, 4), (4, 8, 8), (32, 16, 8), (16, 32, 4), (64, 64, 4), (64, 32, 4),
                               (4, 512, 4), (512, 4, 4), (4, 1024, 4), (1024, 4, 4), (128, 64, 4), (16, 256, 4), (2048, 4, 4),
                               (16, 16, 4), (32, 32, 32), (64, 16, 4), (16, 64, 8), (32, 64, 4), (8, 256, 4)])
def test_two_level_correction_on_any_plane(N, prec, base):
    rng = np.random.default_rng(12)
    with context(opts(N, extra=f"-pc_type fft2 -precision {prec}")) as ctx:
        g = grid_of(ctx.prm)
        mom = [m.astype(np.float32).astype(np.float64) for m in _moments(g, rng, amp=0.1)]
        ctx.set_moments(vlasov_from(mom))
        r = rng.standard_normal(g.nc)
        r -= r.mean()
        z = ctx.pc_apply(r)
        K = list(ctx.prm.kappa_e)
    tol = base + 16 * 2.0 ** -52 * (3 + K[2] ** 2) / (1 - np.cos(2 * np.pi / max(N)))
    ref = orc.pc_apply(g, K, mom[0], r, orc.PC_FFT2)
    z, ref = z - z.mean(), ref - ref.mean()
    assert np.abs(z - ref).max() <= tol * np.abs(ref).max()


# each length of the register four-step passes on each axis (FP64: 16 to 256,
# FP32: to 512), beside lengths of the LDS passes (4, 8); line counts below and
# above a block's 16 to 64 lines.  A mode's symbol is a sum of weights v_o that
# cancels to lambda(k): its roundings, 16 on the two sides, move the mode by
# eps sum|v_o| / |lambda(k)|.  An FP32 transform moves each mode of white noise
# by some eps32 log2(nodes).
@pytest.mark.parametrize("prec,base", [("fp64", 1e-13), ("mixed", 2e-5)])
@pytest.mark.parametrize("extra", ["", "-B0x 1e-5 -B0y 2e-5"])
@pytest.mark.parametrize("N", [(16, 4, 4), (4, 16, 4), (4, 4, 16), (16, 16, 32), (32, 32, 16), (64, 16, 8), (8, 64, 16),
                               (32, 8, 64), (128, 32, 4), (16, 128, 8), (4, 8, 128), (64, 64, 64), (256, 16, 4),
                               (8, 256, 16), (4, 4, 256), (512, 4, 16), (4, 512, 4), (8, 4, 512),
                               # both axes of 16 to 64 points: the plane in one launch
                               (16, 32, 4), (16, 64, 8), (32, 16, 16), (32, 64, 4), (64, 32, 16), (64, 64, 4)])
def test_fft_passes_on_axes_of_any_length(N, extra, prec, base):
    rng = np.random.default_rng(17)
    with context(opts(N, extra=f"-pc_type fft -precision {prec} {extra}")) as ctx:
        g = grid_of(ctx.prm)
        ctx.set_moments(vlasov_from([np.ones(g.nc)] + _moments(g, rng)[1:]))
        r = rng.standard_normal(g.nc)
        r -= r.mean()
        z = ctx.pc_apply(r)
        K = list(ctx.prm.kappa_e)
    delta = np.zeros(g.nc)
    delta[0] = 1
    row = orc.lhs_apply(g, K, np.ones(g.nc), delta)
    lam = np.abs(np.fft.fftn(row.reshape(N[::-1]))).ravel()
    tol = base + 16 * 2.0 ** -52 * np.abs(row).sum() / lam[1:].min()
    ref = orc.pc_apply(g, K, np.ones(g.nc), r, orc.PC_FFT)
    z, ref = z - z.mean(), ref - ref.mean()
    assert np.abs(z - ref).max() <= tol * np.abs(ref).max()


# an iteration's dot products come with A z for at most 8 basis vectors, on grids
# of the column stencil, and are added in the update's kernel where nodes come
# in fours: 12 iterations (past 8 vectors) on node counts that are and are not
# multiples of 4, ragged last blocks, and every kind of row; against a solve
# that takes a second Gram-Schmidt pass, and so sums them in a launch.  Two
# converged solves at this tolerance differ by it times the conditioning of the
# preconditioned operator (below 100), and by the FP64 residual's rounding.
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("N,extra", [((3, 3, 3), "-pc_type jacobi"), ((5, 7, 3), "-pc_type jacobi"),
                                     ((17, 16, 6), "-pc_type zline"), ((17, 15, 9), "-pc_type zline -B0x 1e-5 -B0y 2e-5"),
                                     ((16, 16, 8), "-pc_type fft"), ((32, 32, 32), "-pc_type fft -B0x 1e-5 -B0y 2e-5")])
def test_gmres_dot_products_with_the_operator(N, extra, prec):
    phis = []
    for refine in ("NEVER", "ALWAYS"):
        with context(opts(N, extra=f"{extra} -ksp_rtol 1e-11 -precision {prec} -ksp_max_it 2000 "
                                   f"-ksp_gmres_cgs_refinement_type REFINE_{refine}")) as ctx:
            g = grid_of(ctx.prm)
            ctx.set_moments(vlasov_from(_moments(g, np.random.default_rng(19))))
            phi, st = ctx.solve_potential()
            assert st.converged == 1 and st.residual <= 1e-11, (refine, st.iterations, st.residual)
            phis.append(phi)
    assert np.abs(phis[0] - phis[1]).max() <= 2e-9 * np.abs(phis[1]).max()


# the next direction is launched before the present one's dot products are read,
# except where the cycle, the iteration limit or the expected convergence ends
# it: each end of a cycle against the oracle's iterate after as many steps (in
# exact arithmetic the same; the least-squares step amplifies the rounding of
# the basis by the conditioning of the preconditioned operator, below 100)
@pytest.mark.parametrize("restart", [1, 2, 3, 30])
@pytest.mark.parametrize("max_it", [1, 2, 3, 4, 6])
def test_gmres_cycles_cut_at_any_iteration(restart, max_it):
    N = (16, 16, 8)
    with context(opts(N, extra=f"-pc_type fft -ksp_rtol 1e-14 -ksp_max_it {max_it} -ksp_gmres_restart {restart}")) as ctx:
        g = grid_of(ctx.prm)
        mom = _moments(g, np.random.default_rng(18))
        ctx.set_moments(vlasov_from(mom))
        phi, st = ctx.solve_potential()
        b = ctx.get_rhs()
        K = list(ctx.prm.kappa_e)
    ref, its, conv, _ = orc.solve(g, K, mom[0], b, rtol=1e-14, max_it=max_it, restart=restart)
    assert (st.iterations, st.converged) == (its, 0) and not conv
    assert np.abs(phi - ref).max() <= 1e-11 * np.abs(ref).max()


# columns of 16, 32 and 64 lanes of 1, 2, 4 and 8 planes each, full and ragged,
# and one beyond (513 planes, the levels with x fastest); level widths that are
# and are not multiples of a block's columns.  The level solves are exact but
# reassociated, so FP64 differs from the oracle by roundings that four sweeps
# of each level amplify: the parity test of the cycle allows 1e-10
@pytest.mark.parametrize("prec,tol", [("fp64", 1e-10), ("mixed", 1e-4)])
@pytest.mark.parametrize("N,extra", [((8, 12, 5), ""), ((8, 12, 16), ""), ((12, 8, 17), "-B0x 1e-5 -B0y 2e-5"),
                                     ((20, 12, 33), ""), ((12, 12, 64), "--lhs-type laplacian"), ((12, 8, 65), ""),
                                     ((8, 8, 130), ""), ((8, 4, 300), ""), ((8, 4, 512), ""), ((8, 4, 513), "")])
def test_multigrid_columns_of_any_length(N, extra, prec, tol):
    rng = np.random.default_rng(13)
    with context(opts(N, extra=f"-pc_type mg -precision {prec} {extra}")) as ctx:
        g = grid_of(ctx.prm)
        mom = [m.astype(np.float32).astype(np.float64) for m in _moments(g, rng, amp=0.1)]
        ctx.set_moments(vlasov_from(mom))
        r = rng.standard_normal(g.nc)
        r -= r.mean()
        z = ctx.pc_apply(r)
        K, lt = list(ctx.prm.kappa_e), ctx.prm.lhs_type
    ref = orc.pc_apply(g, K, mom[0], r, orc.PC_MG, lhs_type=lt)
    z, ref = z - z.mean(), ref - ref.mean()
    assert np.abs(z - ref).max() <= tol * np.abs(ref).max()


# the z-line stage in segments: full and ragged columns of each segmentation
# (x-y axes of a power of two, as the preconditioner needs, whose planes here fill
# the blocks' 16 or 32 columns), and the column walk beyond 256 planes;
# B along z (the 2-D correction folded in) and oblique (the plain stage)
@pytest.mark.parametrize("prec,base", [("fp64", 1e-11), ("mixed", 2e-5)])
@pytest.mark.parametrize("extra", ["", "-B0x 1e-5 -B0y 2e-5"])
@pytest.mark.parametrize("N", [(4, 4, 4), (8, 4, 8), (4, 4, 32), (8, 8, 64), (16, 4, 128), (8, 4, 256), (4, 4, 512)])
def test_zline_stage_on_columns_of_any_length(N, extra, prec, base):
    rng = np.random.default_rng(14)
    with context(opts(N, extra=f"-pc_type fft2z -precision {prec} {extra}")) as ctx:
        g = grid_of(ctx.prm)
        mom = [m.astype(np.float32).astype(np.float64) for m in _moments(g, rng, amp=0.1)]
        ctx.set_moments(vlasov_from(mom))
        r = rng.standard_normal(g.nc)
        r -= r.mean()
        z = ctx.pc_apply(r)
        K = list(ctx.prm.kappa_e)
    # the FFT stage's symbol, as in the test of the 2-D correction, and the z-line
    # systems' condition, 2 (1 + K_z^2) / (1 - cos(2 pi / nz)) ulps at most
    tol = base + 16 * 2.0 ** -52 * (3 + K[2] ** 2) / (1 - np.cos(2 * np.pi / max(N)))
    ref = orc.pc_apply(g, K, mom[0], r, orc.PC_FFT2Z)
    z, ref = z - z.mean(), ref - ref.mean()
    assert np.abs(z - ref).max() <= tol * np.abs(ref).max()


# host arrays: one block and its neighbours, many ions on a grid whose Krylov
# basis is too small a scratch for them (one staging piece, and several: 1.2 M
# ions are 91 MB).  The values only change layout (and type, in mixed mode)
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("N,n", [((3, 3, 3), 1), ((4, 5, 6), 257), ((4, 4, 4), 70000), ((12, 10, 11), 1200000)])
def test_ions_survive_the_host_round_trip(N, n, prec):
    rng = np.random.default_rng(15)
    with context(opts(N, extra=f"-precision {prec}"), capacity=n, weighted=True) as ctx:
        p = random_particles(grid_of(ctx.prm), n, rng, weights=True)
        p.pid = rng.permutation(n).astype(np.uint32)
        upload(ctx, p)
        d = ctx.get_particles()
        L = np.array([ctx.prm.L[a] for a in range(3)])
    back = np.argsort(d["pid"])
    want = np.argsort(p.pid)
    assert np.array_equal(d["pid"][back], p.pid[want])
    # mixed: the offset within a cell rounds to FP32 (half an ulp below one, of
    # a cell), velocities and weights to FP32
    tol = 0.0 if prec == "fp64" else 2.0 ** -25 * 1.01
    for a, name in enumerate("xyz"):
        assert np.abs(d[name][back] - getattr(p, name)[want]).max() <= tol * L[a] / N[a] + 4 * 2.0 ** -53 * (tol > 0) * L[a]
    for name in ("vx", "vy", "vz", "w"):
        v = getattr(p, name)[want]
        ref = v if prec == "fp64" else v.astype(np.float32).astype(np.float64)
        assert np.array_equal(d[name][back], ref)


# a potential of 16 MiB and a bit, and its moments, come back in pinned chunks
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("N", [(3, 3, 3), (7, 5, 9), (128, 128, 129)])
def test_grid_arrays_survive_the_host_round_trip(N, prec):
    rng = np.random.default_rng(16)
    with context(opts(N, extra=f"-ksp_gmres_restart 2 -precision {prec}")) as ctx:
        v = rng.standard_normal((ctx.nc, 4))
        ctx.set_moments(v)
        phi = rng.standard_normal(ctx.nc)
        ctx.set_potential(phi)
        assert np.array_equal(ctx.get_moments(), v if prec == "fp64" else v.astype(np.float32).astype(np.float64))
        assert np.array_equal(ctx.get_potential(), phi)


# the FP64 push carries its next ion along: one ion, a wave and its neighbours, a
# block, and several, all in one trip; waves with few and with many colliders
# (nu_in 1e3 and 1e5 s^-1)
@pytest.mark.parametrize("nui", [1e3, 1e5])
@pytest.mark.parametrize("N,n", [((3, 3, 3), 1), ((5, 4, 3), 63), ((5, 4, 3), 65), ((4, 4, 4), 256), ((7, 5, 6), 1023),
                                 ((20, 20, 20), 40000)])
def test_fp64_push_of_any_number_of_ions(N, n, nui):
    rng = np.random.default_rng(17)
    with context(opts(N, extra=f"-nui {nui} -seed 5 --collision-refusal-limit 0 -Np {n}"), capacity=n) as ctx:
        g = grid_of(ctx.prm)
        upload(ctx, random_particles(g, n, rng))
        phi = 0.01 * rng.standard_normal(g.nc)
        ctx.set_potential(phi)
        before = as_particles(ctx.get_particles())
        S = orc.normaliser(before, list(ctx.prm.vn0), ctx.prm.vnT)
        _, P = push_params_of(ctx.prm, step=0)
        st = ctx.update_velocities()
        ctx.update_positions()
        after = as_particles(ctx.get_particles())
    nxt, key, _, _, stats = orc.step(g, P, before, phi, S, list(ctx.prm.E0))
    assert np.array_equal(after.pid, nxt.pid)
    assert (st.accepted, st.refused) == (stats[0], stats[1])
    for a in ("x", "y", "z", "vx", "vy", "vz"):
        assert relmax(getattr(after, a), getattr(nxt, a)) <= 1e-12


# tiles of 4096 cells, 16 a thread: a part of one, one short by a cell, a whole
# one, and further tiles that end within a thread's cells
@pytest.mark.parametrize("N", [(3, 3, 3), (63, 13, 5), (16, 16, 16), (17, 241, 3), (41, 20, 11), (3, 1371, 3)])
def test_cell_offsets_at_the_edges_of_scan_tiles(N):
    rng = np.random.default_rng(20)
    n = 3 * N[0] * N[1] * N[2] + 1
    with context(opts(N), capacity=n) as ctx:
        g = grid_of(ctx.prm)
        p = random_particles(g, n, rng)
        upload(ctx, p)
        got = as_particles(ctx.get_particles())
        v = ctx.collect_moments()
    ps, offs = oracle_sorted(g, p)
    assert np.array_equal(got.pid, ps.pid)
    ref = orc.deposit_sorted(g, ps, offs)
    for a in range(4):
        assert np.array_equal(v[:, a], ref[a])


# ions without a thermal speed: the final speed of a scattering is then more than
# ten times it however small, and every scattering is refused (a drift gives
# them collisions); the oracle divides by zero
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_ions_without_a_thermal_speed_refuse_every_scattering(prec):
    rng = np.random.default_rng(21)
    n = 4000
    with context(opts((6, 5, 4), extra=f"-precision {prec} -Ti 0 -vi0x 500 -nui 1e4 -seed 5 --collision-refusal-limit 0 "
                                       f"-Np {n}"), capacity=n) as ctx:
        assert ctx.prm.viT_r == 0.0
        g = grid_of(ctx.prm)
        upload(ctx, random_particles(g, n, rng))
        phi = 0.01 * rng.standard_normal(g.nc)
        ctx.set_potential(phi)
        before = as_particles(ctx.get_particles())
        S = orc.normaliser(before, list(ctx.prm.vn0), ctx.prm.vnT)
        _, P = push_params_of(ctx.prm, step=0)
        st = ctx.update_velocities()
        after = as_particles(ctx.get_particles())
    nxt, _, _, _, stats = orc.step(g, P, before, phi, S, list(ctx.prm.E0))
    assert stats[0] == 0 and stats[1] > n // 20
    assert st.accepted == 0 and st.refused > n // 20
    if prec == "fp64":
        back, want = np.argsort(after.pid), np.argsort(nxt.pid)
        assert st.refused == stats[1]
        for a in ("vx", "vy", "vz"):
            assert relmax(getattr(after, a)[back], getattr(nxt, a)[want]) <= 1e-12


# mixed: the arrays of up to 6898 ions come in one copy, of more in one each; both
# sides of the line, and a caller that wants some of them.  A copy's latency
# is all that few ions cost, so all four arrays take about what one does
@pytest.mark.parametrize("n", [1, 300, 6898, 6899])
def test_arrays_of_a_few_ions_come_in_one_copy(n):
    rng = np.random.default_rng(22)
    with context(opts((5, 4, 6), extra="-precision mixed"), capacity=n, weighted=True) as ctx:
        p = random_particles(grid_of(ctx.prm), n, rng, weights=True)
        upload(ctx, p)
        d = ctx.get_particles()
        get = chybrid.lib().chy_get_particles
        full = [np.empty((n, 4)), np.empty((n, 4)), np.empty(n), np.empty(n, np.uint32)]
        for want in ((0, 1, 2, 3), (3,), (1,), (0, 2), (1, 3)):
            out = [np.full_like(a, 7) for a in full]
            assert get(ctx._p, *[out[q].ctypes.data if q in want else None for q in range(4)]) == 0
            got = dict(zip(("pos", "vel", "w", "pid"), out))
            for q, name in enumerate(("pos", "vel", "w", "pid")):
                if q not in want:
                    assert (got[name] == 7).all()
                elif q < 2:
                    for a, axis in enumerate("xyz"):
                        assert np.array_equal(got[name][:, a], d[("" if q == 0 else "v") + axis])
                else:
                    assert np.array_equal(got[name], d[name])

        def least(ptrs):
            t = []
            for _ in range(300):
                t0 = time.perf_counter()
                get(ctx._p, *ptrs)
                t.append(time.perf_counter() - t0)
            return min(t)

        if n <= 300:
            all_four = least([a.ctypes.data for a in full])
            one = least([None, None, None, full[3].ctypes.data])
            assert all_four <= 2 * one, (all_four, one)


# many ions on a small grid, with no device memory to be had for their staging (an
# allocator that refuses it, put before the runtime's in a process of its own):
# the ions go in and come back in small pieces
_NO_STAGE = r"""
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
sys.path[:0] = sys.argv[2:5]
import numpy as np
import chybrid
from gpu_cases import context, grid_of, opts, random_particles, upload
n = 30000
for prec in ("fp64", "mixed"):
    with context(opts((4, 4, 4), extra="-precision " + prec), capacity=n, weighted=True) as ctx:
        p = random_particles(grid_of(ctx.prm), n, np.random.default_rng(23), weights=True)
        p.pid = np.arange(n, dtype=np.uint32)[::-1].copy()
        ctypes.c_size_t.in_dll(shim, "fail_from").value = 1
        upload(ctx, p)
        d = ctx.get_particles()
        refused = ctypes.c_size_t.in_dll(shim, "refused").value
        ctypes.c_size_t.in_dll(shim, "fail_from").value = 0
    assert refused > 0
    back, want = np.argsort(d["pid"]), np.argsort(p.pid)
    for name in ("vx", "vy", "vz", "w"):
        v = getattr(p, name)[want]
        assert np.array_equal(d[name][back], v if prec == "fp64" else v.astype(np.float32).astype(np.float64))
    for name in "xyz":
        assert np.abs(d[name][back] - getattr(p, name)[want]).max() <= (0 if prec == "fp64" else 2.0 ** -24 * 0.05)
print("STAGED")
"""


def test_ions_are_staged_without_device_memory_to_spare(tmp_path):
    src, so = tmp_path / "shim.c", tmp_path / "shim.so"
    src.write_text("#include <dlfcn.h>\n#include <stddef.h>\nsize_t fail_from, refused;\n"
                   "int hipMalloc(void **p, size_t n)\n{\n  static int (*next)(void **, size_t);\n"
                   "  if (fail_from && n >= fail_from) { refused++; *p = 0; return 2; }\n"
                   "  if (!next) next = (int (*)(void **, size_t))dlsym(dlopen(\"libamdhip64.so.7\", RTLD_NOW), \"hipMalloc\");\n"
                   "  return next(p, n);\n}\n")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", str(so), str(src), "-ldl"], check=True)
    here = os.path.dirname(os.path.abspath(__file__))
    root = os.path.dirname(here)
    p = subprocess.run([sys.executable, "-c", _NO_STAGE, str(so), here, os.path.join(root, "oracle"),
                        os.path.join(root, "collisional-hybrid_amd")], capture_output=True, text=True, timeout=100)
    assert p.returncode == 0 and "STAGED" in p.stdout, p.stderr[-2000:]


# multigrid takes no more device memory than its z-line factors and its coarse
# levels need: 4 fields of the finest grid and a third of 10 (the coarse levels'
# nodes), with a third of a field and an allocation granule of 2 MiB for each
# array to spare
def test_multigrid_levels_share_the_work_arrays():
    N = (256, 256, 128)
    hip = C.CDLL("libamdhip64.so")
    free, total = C.c_size_t(), C.c_size_t()

    def used(pc):
        assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        before = free.value
        with context(opts(N, extra=f"-pc_type {pc} -ksp_gmres_restart 2"), capacity=1):
            assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
            return before - free.value

    used("jacobi")
    extra = used("mg") - used("jacobi")
    field = 8 * N[0] * N[1] * N[2]
    assert extra <= (4 + 10 / 3 + 1 / 3) * field + 64 * 2 ** 21, extra / field


# the dot products that come with A z (up to 8 basis vectors, iterations 1 to 8) and
# their sums in the update (nodes in fours), against the oracle's iterate after
# as many steps: blocks of columns and groups of planes that are and are not
# whole.  The least-squares step amplifies the basis' rounding, some 100 ulps, by
# the conditioning of the preconditioned operator: 2.3e4 for the first, at most
# 1.2e3 for the others (mixed: 250).  Products that miss one node move an FP64
# iterate by 2e-6 at least, products that miss a plane or a part of a block any
# iterate by 1e-2 (computed with a GMRES that leaves them out).
_DOTS = [((5, 7, 3), "-pc_type jacobi", orc.PC_JACOBI), ((17, 16, 6), "-pc_type zline", orc.PC_ZLINE),
         ((17, 15, 9), "-pc_type zline -B0x 1e-5 -B0y 2e-5", orc.PC_ZLINE), ((16, 16, 8), "-pc_type fft", orc.PC_FFT),
         ((19, 14, 5), "-pc_type jacobi -B0x 1e-5 -B0y 2e-5", orc.PC_JACOBI)]


@pytest.mark.parametrize("refine", ["NEVER", "ALWAYS"])
@pytest.mark.parametrize("N,extra,pc,prec,tol", [(*d, "fp64", 1e-9) for d in _DOTS] + [(*d, "mixed", 2e-3) for d in _DOTS[1:4]])
def test_gmres_iterates_with_the_operators_dot_products(N, extra, pc, prec, tol, refine):
    with context(opts(N, extra=f"{extra} -ksp_rtol 1e-14 -ksp_inner_rtol 1e-7 -precision {prec} "
                               f"-ksp_gmres_cgs_refinement_type REFINE_{refine}")) as ctx:
        g = grid_of(ctx.prm)
        mom = [m.astype(np.float32).astype(np.float64) for m in _moments(g, np.random.default_rng(19))]
        ctx.set_moments(vlasov_from(mom))
        K, b, phis = list(ctx.prm.kappa_e), ctx.compute_rhs(), {}
        for k in (1, 2, 3, 5, 7, 8, 9, 10):
            ctx.set_tolerances(max_it=k)
            ctx.set_potential(np.zeros(g.nc))
            phis[k], st = ctx.solve_potential()
            assert (st.iterations, st.outer) == (k, 1)
    for k, phi in phis.items():
        ref, its, _, _ = orc.solve(g, K, mom[0], b, pc=pc, rtol=1e-14, max_it=k)
        assert its == k
        assert np.abs(phi - ref).max() <= tol * np.abs(ref).max(), k


# the FP64 push's launch holds 2^24 ions: more take several trips, the last one
# partly live, with each trip's ions loaded during the one before
def test_fp64_push_in_several_trips():
    test_fp64_push_of_any_number_of_ions((64, 64, 64), 2 ** 24 + 40003, 1e3)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_push_of_no_ions(prec):
    with context(opts((5, 4, 3), extra=f"-precision {prec} -Np 0"), capacity=8) as ctx:
        none = np.empty(0)
        ctx.set_particles(none, none, none, none, none, none)
        ctx.set_potential(np.random.default_rng(24).standard_normal(ctx.nc))
        st = ctx.update_velocities()
        ctx.update_positions()
        assert (st.accepted, st.refused, ctx.num_particles()) == (0, 0, 0)
        assert not ctx.collect_moments().any()


# the z-line stage on 16 columns where a block takes 32: FP32 columns of 65 to 256
# planes, and the factors of columns beyond 128 planes in both precisions (the
# other blocks take 16 columns, and planes with axes of 4, 8, 16.. nodes hold a
# multiple of 16)
@pytest.mark.parametrize("prec,base", [("fp64", 1e-11), ("mixed", 2e-5)])
@pytest.mark.parametrize("extra", ["", "-B0x 1e-5 -B0y 2e-5"])
@pytest.mark.parametrize("N", [(4, 4, 128), (4, 4, 256)])
def test_zline_stage_in_a_part_of_a_block(N, extra, prec, base):
    test_zline_stage_on_columns_of_any_length(N, extra, prec, base)


# The multigrid of a grid with odd axes is eight sweeps of the z-line smoother on
# one level: in 80 bits, from the operator's rows
def _sweeps80(g, K, n, r):
    nx, ny, nz = (int(v) for v in g.N)
    P, ld = nx * ny, np.longdouble
    D = orc.lhs_dense(g, K, n)
    cols = np.argsort(-np.abs(D), axis=1, kind="stable")[:, :19]
    val = np.take_along_axis(D, cols, 1).astype(ld)
    line = [np.stack([D[np.arange(P) + P * k, np.arange(P) + P * ((k + d) % nz)] for k in range(nz)]).astype(ld)
            for d in (-1, 0, 1)]
    a, b, c = line
    gm = -b[0]
    b = b.copy()
    b[0] -= gm
    b[-1] -= c[-1] * a[0] / gm

    def tri(f):
        cp, y = np.empty_like(f), np.empty_like(f)
        cp[0], y[0] = c[0] / b[0], f[0] / b[0]
        for k in range(1, nz):
            m = b[k] - a[k] * cp[k - 1]
            cp[k], y[k] = c[k] / m, (f[k] - a[k] * y[k - 1]) / m
        for k in range(nz - 2, -1, -1):
            y[k] -= cp[k] * y[k + 1]
        return y

    u = np.zeros((nz, P), ld)
    u[0], u[-1] = gm, c[-1]
    q, x = tri(u), np.zeros(P * nz, ld)
    for _ in range(8):
        y = tri((r - (val * x[cols]).sum(axis=1)).reshape(nz, P))
        y -= (y[0] + a[0] / gm * y[-1]) / (1 + q[0] + a[0] / gm * q[-1]) * q
        x += ld(0.8) * y.ravel()
    return x - x.mean()


# the column factors in segments lose nothing against one plane after another, which
# the oracle does: white noise of 90 % takes the densities of neighbours far
# apart.  The errors of 24 systems in the mean, which a few sums in another order
# move by a quarter at most
@pytest.mark.parametrize("N", [(5, 7, 16), (5, 7, 50), (3, 5, 100)])
def test_column_factors_are_as_accurate_as_the_sequential_ones(N):
    err = {"gpu": [], "oracle": []}
    with context(opts(N, extra="-pc_type mg")) as ctx:
        g = grid_of(ctx.prm)
        K = list(ctx.prm.kappa_e)
        for seed in range(24):
            rng = np.random.default_rng(seed)
            n, r = 1 + 0.9 * rng.uniform(-1, 1, g.nc), rng.standard_normal(g.nc)
            r -= r.mean()
            ctx.set_moments(vlasov_from([n] + 3 * [np.zeros(g.nc)]))
            ref = _sweeps80(g, K, n, r)
            for name, z in (("gpu", ctx.pc_apply(r)), ("oracle", orc.pc_apply(g, K, n, r, orc.PC_MG))):
                err[name].append(float(np.abs(z - z.mean() - ref).max() / np.abs(ref).max()))
    mean = {k: float(np.exp(np.mean(np.log(v)))) for k, v in err.items()}
    assert mean["gpu"] <= 1.25 * mean["oracle"], mean


# mixed, z axes of 16 to 128 points: a mode is divided by its symbol in FP64.  The
# gain of each mode of the Laplacian whose symbol is within a factor 4 of the
# largest, averaged over 400 draws of white noise in these modes, against that
# on a grid with 1.3 times the spacing: the gains of the transforms, which their
# rounded twiddles make, are the same.  Roundings of the transforms, some 2e-7 of a
# mode, leave 2e-7 sqrt(2 / 400) = 1.4e-8 in the mean square over the modes;
# quotients in FP32 (the symbol, its reciprocal, the scale and the product, each
# 2^-24 at most) leave 2^-24 / sqrt(3) sqrt(2 x 4 / 2) or more than 5e-8
@pytest.mark.parametrize("N", [(16, 16, 16), (16, 8, 32), (8, 8, 64), (8, 8, 128)])
def test_mixed_fft_divides_by_the_symbol_in_fp64(N):
    rng = np.random.default_rng(25)
    shape = N[::-1]
    gains = []
    delta = np.zeros(int(np.prod(N)))
    delta[0] = 1
    noise = None
    for spacing in (0.05, 0.065):
        with context(opts(N, L=spacing, extra="-pc_type fft -precision mixed --lhs-type laplacian")) as ctx:
            g = grid_of(ctx.prm)
            row = orc.lhs_apply(g, list(ctx.prm.kappa_e), np.ones(g.nc), delta, lhs_type=ctx.prm.lhs_type)
            lam = np.fft.fftn(row.reshape(shape)).real
            if noise is None:
                band = np.abs(lam) >= np.abs(lam).max() / 4
                noise = [np.fft.ifftn(np.fft.fftn(rng.standard_normal(shape)) * band).real.astype(np.float32)
                         for _ in range(400)]
            ctx.set_moments(vlasov_from([np.ones(g.nc)] + 3 * [np.zeros(g.nc)]))
            num, den = 0.0, 0.0
            for r in noise:
                R = np.fft.fftn(r.astype(np.float64))
                Z = np.fft.fftn(ctx.pc_apply(r.astype(np.float64).ravel()).reshape(shape))
                num, den = num + (Z * R.conj()).real, den + np.abs(R) ** 2
            gains.append((num / np.where(band, den, 1) * lam)[band])
    assert np.sqrt(np.mean(np.square(gains[0] / gains[1] - 1))) <= 2.8e-8


# a small field comes back in the time of one blocking copy
def test_a_small_field_comes_back_in_one_blocking_copy():
    def least(f):
        t = []
        for _ in range(300):
            t0 = time.perf_counter()
            assert f() == 0
            t.append(time.perf_counter() - t0)
        return min(t)

    hip = C.CDLL("libamdhip64.so")
    with context(opts((8, 8, 8)), capacity=1) as ctx:
        phi, out, dev = np.random.default_rng(26).standard_normal(ctx.nc), np.empty(ctx.nc), C.c_void_p()
        ctx.set_potential(phi)
        assert hip.hipMalloc(C.byref(dev), C.c_size_t(out.nbytes)) == 0
        try:
            copy = least(lambda: hip.hipMemcpy(C.c_void_p(out.ctypes.data), dev, C.c_size_t(out.nbytes), 2))
        finally:
            hip.hipFree(dev)
        get = least(lambda: chybrid.lib().chy_get_potential(ctx._p, out.ctypes.data))
        assert np.array_equal(out, phi)
    assert get <= 1.4 * copy, (get, copy)


# the 2-D correction makes one Gram-Schmidt pass, the oracle two: in each of its
# forms (planes in registers, in LDS and by launches) on densities that leave the
# second direction nothing but rounding, and on one that varies twentyfold in x
# and y; tolerances as in the test of any plane
@pytest.mark.parametrize("prec,base", [("fp64", 1e-12), ("mixed", 2e-5)])
@pytest.mark.parametrize("contrast", [0.0, 0.001, 0.95])
@pytest.mark.parametrize("N", [(16, 16, 8), (8, 64, 8), (64, 64, 4)])
def test_two_level_correction_at_any_contrast(N, contrast, prec, base):
    rng = np.random.default_rng(27)
    with context(opts(N, extra=f"-pc_type fft2 -precision {prec}")) as ctx:
        g = grid_of(ctx.prm)
        wave = np.sin(2 * np.pi * np.arange(N[0]) / N[0]) * np.cos(2 * np.pi * np.arange(N[1]) / N[1])[:, None]
        n = (1 + contrast * np.broadcast_to(wave, N[::-1]).ravel()).astype(np.float32).astype(np.float64)
        ctx.set_moments(vlasov_from([n] + 3 * [np.zeros(g.nc)]))
        r = rng.standard_normal(g.nc)
        r -= r.mean()
        z = ctx.pc_apply(r)
        K = list(ctx.prm.kappa_e)
    tol = base + 16 * 2.0 ** -52 * (3 + K[2] ** 2) / (1 - np.cos(2 * np.pi / max(N)))
    ref = orc.pc_apply(g, K, n, r, orc.PC_FFT2)
    z, ref = z - z.mean(), ref - ref.mean()
    assert np.abs(z - ref).max() <= tol * np.abs(ref).max()
