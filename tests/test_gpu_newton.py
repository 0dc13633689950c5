"""GPU parity of NewtonInverse against the CPU oracle and closed forms."""
import numpy as np
import pytest
import torch

import oracle
from lfcheck import TORCH_DT, assert_newton_close, gen

pytestmark = pytest.mark.gpu


def gram(bh, n, d, seed, shift=1e-3, scale=1.0):
    """A = exp(-L1(k_i, k_j) / sqrt(d)) + shift*I from k ~ N(0, scale^2) (BASELINE config recipe)."""
    k = gen((1, bh, n, d), seed, "f64", scale=scale)
    D = oracle.laplace_forward(k, k.transpose(-1, -2).contiguous(), "f64")[0]
    return np.exp(-D / np.sqrt(d)) + shift * np.eye(n)


NS = [1, 5, 16, 17, 32, 48, 49, 64, 65, 80, 96, 100, 112, 113, 128]


@pytest.mark.parametrize("n", NS)
@pytest.mark.parametrize("iters", [0, 1, 10])
def test_newton_forward_f32(gpu, n, iters):
    import laplacianformer_amd as lf

    print(f"newton forward n={n} iters={iters}", flush=True)
    A = torch.from_numpy(gram(6, n, 32, seed=n)).float().reshape(2, 3, n, n)
    out = torch.empty_like(A, device=gpu)
    lf.ext().NewtonInverse_forward(A.to(gpu), out, iters)
    ref = oracle.newton_forward(A, iters, "f32")
    assert_newton_close(out, ref, "f32", f"n={n} it={iters}")


@pytest.mark.parametrize("dt", ["f16", "bf16", "f64"])
@pytest.mark.parametrize("n", [16, 49, 64, 96])
def test_newton_forward_dtypes(gpu, dt, n):
    import laplacianformer_amd as lf

    print(f"newton forward {dt} n={n}", flush=True)
    A = torch.from_numpy(gram(4, n, 64, seed=100 + n)).reshape(2, 2, n, n).to(TORCH_DT[dt])
    out = torch.empty_like(A, device=gpu)
    lf.ext().NewtonInverse_forward(A.to(gpu), out, 10)
    ref = oracle.newton_forward(A, 10, dt)
    assert_newton_close(out, ref, dt, f"{dt} n={n}", rtol=1e-4 if dt != "f64" else 1e-10)


@pytest.mark.parametrize("dt", ["f32", "f16", "bf16", "f64"])
@pytest.mark.parametrize("n", [1, 16, 17, 49, 64, 65, 96, 128])
def test_newton_backward(gpu, dt, n):
    import laplacianformer_amd as lf

    print(f"newton backward {dt} n={n}", flush=True)
    V = gen((2, 2, n, n), 7 + n, dt, scale=0.3)
    G = gen((2, 2, n, n), 8 + n, dt)
    out = torch.empty_like(V, device=gpu)
    if dt == "f64" and n > 96:
        # Outside the fp64 envelope (two fp64 n x n buffers per workgroup in LDS):
        # the documented rejection, before any launch.
        with pytest.raises(RuntimeError, match="fp64"):
            lf.ext().NewtonInverse_backward(G.to(gpu), V.to(gpu), out)
        return
    lf.ext().NewtonInverse_backward(G.to(gpu), V.to(gpu), out)
    ref = oracle.newton_backward(G, V, dt)
    assert_newton_close(out, ref, dt, f"bwd {dt} n={n}", rtol=1e-5 if dt != "f64" else 1e-12)


def test_newton_backward_not_square(gpu):
    """A non-square inverse is rejected before any launch (the kernels would read
    and write B*H*N*N elements of [B, H, N, K] tensors)."""
    import laplacianformer_amd as lf

    V = torch.zeros((1, 2, 8, 5), device=gpu)
    G = torch.zeros((1, 2, 8, 5), device=gpu)
    out = torch.empty((1, 2, 8, 5), device=gpu)
    with pytest.raises(RuntimeError, match="last two dims of inverse must be equal"):
        lf.ext().NewtonInverse_backward(G, V, out)


def test_newton_config3(gpu):
    """1024 matrices 64x64 fp32, 12 iterations, forward + backward."""
    import laplacianformer_amd as lf

    print("newton config 3", flush=True)
    A = torch.from_numpy(gram(1024, 64, 64, seed=1003)).float().reshape(1024, 1, 64, 64)
    G = gen((1024, 1, 64, 64), 1013, "f32")
    Ad, Gd = A.to(gpu), G.to(gpu)
    V = torch.empty_like(Ad)
    dA = torch.empty_like(Ad)
    lf.ext().NewtonInverse_forward(Ad, V, 12)
    lf.ext().NewtonInverse_backward(Gd, V, dA)
    ref = oracle.newton_forward(A, 12, "f32")
    assert_newton_close(V, ref, "f32", "cfg3 fwd")
    assert_newton_close(dA, oracle.newton_backward(G, V.cpu(), "f32"), "f32", "cfg3 bwd", rtol=1e-5)
    # Residual ||P X - I||_F matches the oracle's within 1e-4 * sqrt(n).
    P = A.double() + 0.01 * torch.eye(64, dtype=torch.float64)
    r_gpu = torch.linalg.matrix_norm(P @ V.cpu().double() - torch.eye(64, dtype=torch.float64))
    r_ref = torch.linalg.matrix_norm(P @ torch.from_numpy(ref).double() - torch.eye(64, dtype=torch.float64))
    assert (r_gpu - r_ref).abs().max().item() <= 1e-4 * 8


@pytest.mark.parametrize("bh", [257, 600, 1000, 2048])
def test_newton_backward_persistent(gpu, bh):
    """Full 64 x 64 fp32 matrices at 2 to 8 per CU take the persistent backward (one
    workgroup per CU, its matrices through four LDS slots in turn); counts that leave
    the last workgroup short, against the oracle."""
    import laplacianformer_amd as lf

    print(f"newton backward persistent bh={bh}", flush=True)
    V = gen((bh, 1, 64, 64), 40 + bh, "f32", scale=0.3)
    G = gen((bh, 1, 64, 64), 41 + bh, "f32")
    out = torch.empty_like(V, device=gpu)
    lf.ext().NewtonInverse_backward(G.to(gpu), V.to(gpu), out)
    assert_newton_close(out, oracle.newton_backward(G, V, "f32"), "f32", f"bwd persistent bh={bh}", rtol=1e-5)


@pytest.mark.parametrize("case", ["symmetric", "one_pair", "general"])
@pytest.mark.parametrize("bh", [3, 600])
def test_newton_forward_n49_symmetry(gpu, case, bh):
    """fp32 n = 49 runs the symmetric iteration (upper tiles, mirrored) when P is exactly
    symmetric and the general one otherwise, decided per matrix in the kernel. Both against
    the oracle; the symmetric path's result is exactly symmetric, a matrix with a single
    asymmetric pair and a general matrix take the general path. 600 matrices: two waves per
    strip (the 8-wave variant of the symmetric body)."""
    import laplacianformer_amd as lf

    print(f"newton forward n=49 {case} bh={bh}", flush=True)
    n = 49
    A = gram(bh, n, 64, seed=300 + bh)
    if case == "one_pair":
        A[:, 3, 40] += 1e-3  # every matrix asymmetric in one element pair
    elif case == "general":
        A = A + 1e-4 * np.random.default_rng(7).standard_normal(A.shape)
    At = torch.from_numpy(A).float().reshape(bh, 1, n, n)
    out = torch.empty_like(At, device=gpu)
    lf.ext().NewtonInverse_forward(At.to(gpu), out, 10)
    ref = oracle.newton_forward(At, 10, "f32")
    assert_newton_close(out, ref, "f32", f"n=49 {case}", rtol=1e-4)
    o = out.cpu()
    if case == "symmetric":
        assert torch.equal(o, o.transpose(-1, -2)), "symmetric path result not exactly symmetric"


def test_newton_closed_forms(gpu):
    """Diagonal A = c I: X_k = (1 - (-0.8)^(2^k)) / mu * I with mu = c + 0.01; and iter = 0 gives alpha P."""
    import laplacianformer_amd as lf

    for n, c in ((16, 0.5), (49, 2.0), (128, 0.09)):
        mu = c + 0.01
        A = (c * torch.eye(n)).reshape(1, 1, n, n).repeat(2, 1, 1, 1)
        for k in (0, 1, 3, 6):
            out = torch.empty_like(A, device=gpu)
            lf.ext().NewtonInverse_forward(A.to(gpu), out, k)
            expect = (1 - (-0.8) ** (2 ** k)) / mu
            d = torch.diagonal(out.cpu().double(), dim1=-2, dim2=-1)
            assert torch.allclose(d, torch.full_like(d, expect), rtol=2e-6), (n, c, k)
            off = out.cpu().double() - torch.diag_embed(d)
            assert off.abs().max().item() == 0.0


def test_newton_errors(gpu):
    import laplacianformer_amd as lf

    L = lf.ext()
    A = torch.zeros((1, 1, 257, 257), device=gpu)
    with pytest.raises(RuntimeError, match="N=257 is not supported"):
        L.NewtonInverse_forward(A, torch.empty_like(A), 3)
    with pytest.raises(RuntimeError, match="must be 4D"):
        L.NewtonInverse_forward(torch.zeros((3, 4, 4), device=gpu), torch.empty((3, 4, 4), device=gpu), 3)
    with pytest.raises(RuntimeError, match="same shape"):
        L.NewtonInverse_forward(torch.zeros((1, 1, 4, 4), device=gpu), torch.empty((1, 1, 5, 5), device=gpu), 3)
    assert L.NewtonInverse_is_supported(256) and not L.NewtonInverse_is_supported(257)
    assert not L.NewtonInverse_is_supported(0)


def test_newton_autograd(gpu):
    import laplacianformer_amd as lf

    A = torch.from_numpy(gram(2, 49, 32, seed=4)).float().reshape(1, 2, 49, 49)
    Ad = A.to(gpu).requires_grad_()
    V = lf.newton_inverse(Ad, 10)
    G = gen((1, 2, 49, 49), 5, "f32")
    V.backward(G.to(gpu))
    assert_newton_close(V, oracle.newton_forward(A, 10), "f32")
    assert_newton_close(Ad.grad, oracle.newton_backward(G, V.detach().cpu()), "f32", rtol=1e-5)


def test_newton_golden_closed_form(gpu):
    """tests/golden/newton_closed.npz: eigen closed form of the iteration with the reference init."""
    import os

    import laplacianformer_amd as lf

    z = np.load(os.path.join(os.path.dirname(__file__), "golden", "newton_closed.npz"))
    for n in (5, 49, 64, 136):
        A = torch.from_numpy(z[f"A_{n}"]).float().reshape(1, 1, n, n)
        for it in (0, 1, 4, 10):
            out = torch.empty_like(A, device=gpu)
            lf.ext().NewtonInverse_forward(A.to(gpu), out, it)
            assert_newton_close(out, z[f"X_{n}_{it}"][None, None], "f32", f"closed n={n} it={it}")


# ---- 128 < n <= 256: batched-GEMM path (beyond the reference's n <= 128) ----

@pytest.mark.parametrize("n", [129, 130, 192, 200, 256])
@pytest.mark.parametrize("iters", [0, 1, 10])
def test_newton_large_forward_f32(gpu, n, iters):
    import laplacianformer_amd as lf

    print(f"newton large forward n={n} iters={iters}", flush=True)
    A = torch.from_numpy(gram(3, n, 32, seed=n)).float().reshape(3, 1, n, n)
    out = torch.empty_like(A, device=gpu)
    lf.ext().NewtonInverse_forward(A.to(gpu), out, iters)
    assert_newton_close(out, oracle.newton_forward(A, iters, "f32"), "f32", f"n={n} it={iters}")


@pytest.mark.parametrize("dt", ["f16", "bf16"])
def test_newton_large_forward_dtypes(gpu, dt):
    import laplacianformer_amd as lf

    n = 200
    print(f"newton large forward {dt} n={n}", flush=True)
    A = torch.from_numpy(gram(2, n, 64, seed=300)).reshape(1, 2, n, n).to(TORCH_DT[dt])
    out = torch.empty_like(A, device=gpu)
    lf.ext().NewtonInverse_forward(A.to(gpu), out, 10)
    assert_newton_close(out, oracle.newton_forward(A, 10, dt), dt, f"{dt} n={n}")


@pytest.mark.parametrize("dt", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("n", [129, 200, 256])
def test_newton_large_backward(gpu, dt, n):
    import laplacianformer_amd as lf

    print(f"newton large backward {dt} n={n}", flush=True)
    V = gen((2, 1, n, n), 17 + n, dt, scale=0.1)
    G = gen((2, 1, n, n), 18 + n, dt)
    out = torch.empty_like(V, device=gpu)
    lf.ext().NewtonInverse_backward(G.to(gpu), V.to(gpu), out)
    assert_newton_close(out, oracle.newton_backward(G, V, dt), dt, f"bwd {dt} n={n}", rtol=1e-5)


def test_newton_large_backward_in_place_and_unaligned(gpu):
    """fp32 n = 256 reads and writes the caller's tensors directly unless the output
    overlaps the inverse or a pointer is not 16-byte aligned; every route gives the
    same bits."""
    import laplacianformer_amd as lf

    n = 256
    print("newton large backward aliasing / alignment", flush=True)
    V = gen((2, 1, n, n), 41, "f32", scale=0.1).to(gpu)
    G = gen((2, 1, n, n), 42, "f32").to(gpu)
    L = lf.ext()
    want = torch.empty_like(V)
    L.NewtonInverse_backward(G, V, want)
    got = V.clone()
    L.NewtonInverse_backward(G, got, got)  # output written over the inverse
    assert torch.equal(got, want)
    buf = torch.empty(3 * V.numel() + 1, device=gpu)
    Vu = buf[1:1 + V.numel()].view_as(V).copy_(V)  # 4-byte offset: not 16-byte aligned
    Gu = buf[1 + V.numel():1 + 2 * V.numel()].view_as(G).copy_(G)
    Ou = buf[1 + 2 * V.numel():].view_as(V)
    L.NewtonInverse_backward(Gu, Vu, Ou)
    assert torch.equal(Ou, want)
    A = torch.from_numpy(gram(1, n, 32, seed=5)).float().reshape(1, 1, n, n).to(gpu)
    fa = torch.empty_like(A)
    L.NewtonInverse_forward(A, fa, 3)
    fb = torch.empty(A.numel() + 1, device=gpu)[1:].view_as(A)
    L.NewtonInverse_forward(A, fb, 3)
    assert torch.equal(fa, fb)


def test_newton_large_closed_form(gpu):
    """Diagonal A = c I at n = 256: X_k = (1 - (-0.8)^(2^k)) / (c + 0.01) * I, off-diagonal exactly 0."""
    import laplacianformer_amd as lf

    n, c = 256, 0.3
    mu = c + 0.01
    A = (c * torch.eye(n)).reshape(1, 1, n, n)
    for k in (0, 2, 5):
        out = torch.empty_like(A, device=gpu)
        lf.ext().NewtonInverse_forward(A.to(gpu), out, k)
        d = torch.diagonal(out.cpu().double(), dim1=-2, dim2=-1)
        assert torch.allclose(d, torch.full_like(d, (1 - (-0.8) ** (2 ** k)) / mu), rtol=2e-6), k
        assert (out.cpu().double() - torch.diag_embed(d)).abs().max().item() == 0.0


def test_newton_config4(gpu):
    """BASELINE config 4 (Newton part): 128 Gram matrices 256x256 fp32, 16 iterations, fwd + bwd."""
    import laplacianformer_amd as lf

    print("newton config 4", flush=True)
    A = torch.from_numpy(gram(128, 256, 64, seed=1004, scale=0.5)).float().reshape(16, 8, 256, 256)
    G = gen((16, 8, 256, 256), 1014, "f32")
    Ad, Gd = A.to(gpu), G.to(gpu)
    V = torch.empty_like(Ad)
    dA = torch.empty_like(Ad)
    lf.ext().NewtonInverse_forward(Ad, V, 16)
    lf.ext().NewtonInverse_backward(Gd, V, dA)
    ref = oracle.newton_forward(A, 16, "f32")
    assert_newton_close(V, ref, "f32", "cfg4 fwd")
    assert_newton_close(dA, oracle.newton_backward(G, V.cpu(), "f32"), "f32", "cfg4 bwd", rtol=1e-5)


@pytest.mark.parametrize("bh,n,dt", [(511, 64, "f32"), (512, 64, "f32"), (513, 50, "f32"), (515, 63, "f16"),
                                     (3, 33, "f32"), (2, 47, "bf16"), (2, 81, "f32"), (2, 97, "bf16"), (2, 127, "f16")])
@pytest.mark.parametrize("iters", [0, 1, 2, 9])
def test_newton_forward_split(gpu, bh, n, dt, iters):
    """The bf16-piece iterations at the edges of their size and count rules: two matrices to a
    workgroup (512 and more of 48 < n <= 64, an odd last one), one 16-column strip per wave
    (fewer), one workgroup per matrix above 64; general matrices, whose iterates are not
    symmetric, so that a transposed tile would show."""
    import laplacianformer_amd as lf

    print(f"newton forward split bh={bh} n={n} {dt} iters={iters}", flush=True)
    A = gram(1, n, 64, seed=900 + n)
    noise = gen((bh, n, n), 901 + n, "f64").numpy()
    A = torch.from_numpy(A + 1e-2 / n * noise).reshape(bh, 1, n, n).to(TORCH_DT[dt])
    out = torch.full_like(A, float("nan"), device=gpu)
    lf.ext().NewtonInverse_forward(A.to(gpu), out, iters)
    assert_newton_close(out, oracle.newton_forward(A, iters, dt), dt, f"bh={bh} n={n} {dt} it={iters}")


@pytest.mark.parametrize("bh,n,dt,iters", [(3, 17, "f32", 9), (513, 17, "f32", 5), (513, 17, "bf16", 5),
                                           (512, 32, "f32", 5), (513, 32, "f16", 3), (513, 30, "f32", 2),
                                           (512, 50, "bf16", 1), (512, 50, "bf16", 2), (511, 50, "f32", 2),
                                           (2, 65, "f32", 9), (513, 65, "f32", 3), (2, 65, "bf16", 9),
                                           (256, 80, "f32", 2), (257, 80, "f16", 2), (257, 90, "bf16", 3),
                                           (2, 105, "bf16", 6), (2, 105, "f16", 0), (2, 128, "f32", 2),
                                           (65, 128, "f32", 3), (64, 128, "f16", 3), (256, 128, "f32", 4),
                                           (256, 115, "bf16", 5), (3, 33, "f32", 6), (513, 33, "f32", 3),
                                           (3, 33, "bf16", 6), (600, 24, "bf16", 6), (769, 24, "f32", 4),
                                           (512, 64, "f32", 2), (512, 64, "bf16", 2), (2, 90, "f32", 1),
                                           (257, 80, "f32", 3), (257, 96, "f32", 3), (2, 105, "bf16", 1)])
def test_newton_forward_fp32_rule(gpu, bh, n, dt, iters):
    """Both sides of the rule between the fp32 matrix instructions and the bf16 pieces (counts of
    matrices and iterations, n = 17 and 65), on general matrices."""
    import laplacianformer_amd as lf

    print(f"newton forward rule bh={bh} n={n} {dt} iters={iters}", flush=True)
    noise = gen((bh, n, n), 921 + n, "f64").numpy()
    A = torch.from_numpy(gram(1, n, 64, seed=920 + n) + 1e-2 / n * noise).reshape(bh, 1, n, n).to(TORCH_DT[dt])
    out = torch.full_like(A, float("nan"), device=gpu)
    lf.ext().NewtonInverse_forward(A.to(gpu), out, iters)
    assert_newton_close(out, oracle.newton_forward(A, iters, dt), dt, f"bh={bh} n={n} {dt} it={iters}")


@pytest.mark.parametrize("bh,n", [(5, 40), (5, 64), (601, 64), (5, 100), (5, 128), (9, 196), (9, 256)])
def test_newton_forward_split_nonfinite(gpu, bh, n):
    """A matrix with a NaN or an infinity gives no finite value after an iteration (every row
    and column of the products meets it); the other matrices of the batch are untouched. Matrices
    0 and 3 are the bad ones: where two matrices share a workgroup (601 of them) each has a good
    neighbour, once behind it and once before."""
    import laplacianformer_amd as lf

    print(f"newton forward non-finite bh={bh} n={n}", flush=True)
    A = torch.from_numpy(gram(bh, n, 64, seed=950 + n)).float().reshape(bh, 1, n, n)
    bad = A.clone()
    bad[0, 0, 3, 5] = float("nan")
    bad[3, 0, n - 1, 2] = float("inf")
    good, got = torch.empty_like(A, device=gpu), torch.empty_like(A, device=gpu)
    lf.ext().NewtonInverse_forward(A.to(gpu), good, 3)
    lf.ext().NewtonInverse_forward(bad.to(gpu), got, 3)
    assert not torch.isfinite(got[[0, 3]]).any()
    rest = [i for i in range(bh) if i not in (0, 3)]
    assert len(rest) >= 3 and torch.isfinite(good[rest]).all()
    assert torch.equal(got[rest], good[rest])


@pytest.mark.parametrize("bh,n", [(3, 16), (3, 30), (771, 30), (3, 40), (3, 64), (600, 64), (3, 100), (3, 128)])
def test_newton_forward_range(gpu, bh, n):
    """The largest finite entries (above the largest bf16) and a huge matrix: alpha underflows to 0
    and every iterate is 0, no infinity or NaN; without an iteration alpha P itself, its
    infinities included. The other matrices of the batch are untouched."""
    import laplacianformer_amd as lf

    print(f"newton forward range bh={bh} n={n}", flush=True)
    A = torch.from_numpy(gram(bh, n, 64, seed=960 + n)).float().reshape(bh, 1, n, n)
    big = A.clone()
    big[0, 0, 1, n - 2] = torch.finfo(torch.float32).max
    big[1] *= 2.0 ** 126
    good, got = torch.empty_like(A, device=gpu), torch.empty_like(A, device=gpu)
    lf.ext().NewtonInverse_forward(A.to(gpu), good, 7)
    lf.ext().NewtonInverse_forward(big.to(gpu), got, 7)
    assert not got[:2].any() and torch.equal(got[2:], good[2:]) and bh > 2
    big = A.clone()
    big[0, 0, 2, 3] = float("-inf")
    lf.ext().NewtonInverse_forward(big.to(gpu), got, 0)
    ref = oracle.newton_forward(big, 0, "f32")
    assert ref[0, 0, 2, 3] == -np.inf and got[0, 0, 2, 3].item() == -np.inf
    ref[0, 0, 2, 3] = got[0, 0, 2, 3] = 0.0
    assert_newton_close(got, ref, "f32", f"n={n} it=0")


@pytest.mark.parametrize("bh,n", [(64, 256), (65, 196), (3, 193), (9, 150)])
def test_newton_large_split(gpu, bh, n):
    """The piece products of n > 128 on both tile sizes (128 x 128 where they give every CU one),
    on general matrices (no symmetric iterate) and gradients; matrix counts off a multiple of 8."""
    import laplacianformer_amd as lf

    print(f"newton large split bh={bh} n={n}", flush=True)
    A = gram(1, n, 64, seed=970 + n) + 1e-2 / n * gen((bh, n, n), 971 + n, "f64").numpy()
    A = torch.from_numpy(A).float().reshape(bh, 1, n, n)
    out = torch.empty_like(A, device=gpu)
    lf.ext().NewtonInverse_forward(A.to(gpu), out, 3)
    assert_newton_close(out, oracle.newton_forward(A, 3, "f32"), "f32", f"bh={bh} n={n}")
    V, G = gen((bh, 1, n, n), 972 + n, "f32", scale=0.3), gen((bh, 1, n, n), 973 + n, "f32")
    lf.ext().NewtonInverse_backward(G.to(gpu), V.to(gpu), out)
    assert_newton_close(out, oracle.newton_backward(G, V, "f32"), "f32", f"bwd bh={bh} n={n}", rtol=1e-5)


@pytest.mark.parametrize("bh,n", [(64, 256), (3, 192), (3, 150)])
@pytest.mark.parametrize("ev,eg", [(0, -120), (0, -146), (0, 127), (60, 7), (-60, -10), (-130, 120), (80, -140)])
def test_newton_large_backward_range(gpu, bh, n, ev, eg):
    """n > 128: inverses and gradients of any magnitude (V ~ 2^ev, G ~ 2^eg; another batch entry
    stays of order 1) give what the fp64 products give wherever that is a float: the pieces
    hold no subnormal tail and no infinity of their own."""
    import laplacianformer_amd as lf

    print(f"newton large backward range bh={bh} n={n} ev={ev} eg={eg}", flush=True)
    V, G = gen((bh, 1, n, n), 982 + n, "f32", scale=0.05), gen((bh, 1, n, n), 983 + n, "f32", scale=0.1)
    V[1:], G[1:] = torch.ldexp(V[1:], torch.tensor(ev)), torch.ldexp(G[1:].clamp(-1, 1), torch.tensor(eg))
    out = torch.full_like(V, float("nan"), device=gpu)
    lf.ext().NewtonInverse_backward(G.to(gpu), V.to(gpu), out)
    v64, g64 = V[:3, 0].double(), G[:3, 0].double()
    ref = -(v64.mT @ g64 @ v64.mT)
    got = out[:3, 0].cpu().double()
    assert torch.isfinite(got).all()
    for i in range(3):
        # 1e-5 of the largest entry, as elsewhere, and half a subnormal unit at the store.
        lim = 1e-5 * ref[i].abs().max() + 2.0 ** -150
        assert ((got[i] - ref[i]).abs() <= lim).all(), (i, ((got[i] - ref[i]).abs().max() / ref[i].abs().max()).item())


@pytest.mark.parametrize("bh,n", [(64, 256), (3, 192), (3, 150)])
@pytest.mark.parametrize("ev,eg", [(0, -120), (0, -146), (0, 127), (60, 7), (-95, 80), (-100, 120), (40, -140)])
def test_newton_large_backward_range(gpu, bh, n, ev, eg):
    """n > 128: inverses and gradients of any magnitude (V ~ 2^ev, G ~ 2^eg in all but the first
    matrix) keep fp32 accuracy: the pieces lose no low bits and no finite entry."""
    import laplacianformer_amd as lf

    print(f"newton large backward range bh={bh} n={n} ev={ev} eg={eg}", flush=True)
    V, G = gen((bh, 1, n, n), 982 + n, "f32", scale=0.05), gen((bh, 1, n, n), 983 + n, "f32", scale=0.1)
    V[1:], G[1:] = torch.ldexp(V[1:], torch.tensor(ev)), torch.ldexp(G[1:].clamp(-1, 1), torch.tensor(eg))
    out = torch.full_like(V, float("nan"), device=gpu)
    lf.ext().NewtonInverse_backward(G.to(gpu), V.to(gpu), out)
    v64, g64 = V[:3, 0].double(), G[:3, 0].double()
    ref = -(v64.mT @ g64 @ v64.mT)
    got = out[:3, 0].cpu().double()
    assert torch.isfinite(got).all()
    for i in range(3):
        # 1e-5 of the largest entry, as elsewhere; S = V^T G is an fp32 tensor, whose subnormals
        # end at 2^-149: half a unit per term of the second sum.
        lim = 1e-5 * ref[i].abs().max() + 2.0 ** -150 * v64[i].abs().sum(1).max()
        assert ((got[i] - ref[i]).abs() <= lim).all(), (i, ((got[i] - ref[i]).abs().max() / ref[i].abs().max()).item())
