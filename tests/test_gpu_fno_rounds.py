"""GPU: the surrogate's persistent kernels where a workgroup takes several rounds
(the other tests' sizes give it one), and the DFTs at contractions past 64.

On an MI355X a launch of k_column holds at most 512 workgroups of two or four
per CU, of one point each past 128 times and of two up to 128, and k_wgrad 512
of 256 points, so the sizes here give from three rounds to nine, the next one
loaded under the present one and, in the columns, written in place.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,B,X,Y,T,mx,my,mt,H", [
    (32, 2, 40, 40, 160, 8, 8, 16, 64),
    # two points a group, an odd number of points: the last group repeats one
    (16, 3, 47, 45, 33, 6, 4, 7, 32),
    # the wide form (one workgroup per CU), whose training head is separate
    (64, 1, 48, 47, 130, 4, 6, 9, 64),
    (8, 2, 63, 61, 20, 4, 4, 5, 64)])
def test_fused_kernels_over_several_rounds(gpu_lib, W, B, X, Y, T, mx, my, mt, H):
    """the fused forward and backward against the separate kernels: every saved
    tensor, the prediction and the mode weights' gradients are the same bits;
    the inference form within 1e-4 of the change the network makes; the other
    gradients, FP32 sums of K = B X Y T terms in another order, round by about
    2^-24 sqrt(K) of a sum of size sqrt(K), at most 4.3e-5 here: within 1e-4 of
    the largest"""
    from mpc_amd.fno import DArr, FnoConfig, FnoGpu, init_params
    print(f"case rounds W={W} B={B} X={X} Y={Y} T={T} modes={mx},{my},{mt} H={H}", flush=True)
    assert 2.0 ** -24 * np.sqrt(B * X * Y * T) <= 4.3e-5
    cfg = FnoConfig(X=X, Y=Y, T=T, width=W, layers=3, mx=mx, my=my, mt=mt, hidden=H)
    p = init_params(cfg, seed=W + T)
    rng = np.random.default_rng(T)
    for k in p:
        if k[0] == "R":
            p[k] *= W
        if k[0] in "bq":
            p[k] = 0.1 * rng.standard_normal(p[k].shape)
    x = rng.standard_normal((B, cfg.cin, X, Y, T)).astype(np.float32)
    dx, tgt = DArr.of(x), DArr.of(rng.standard_normal((B, 2, X, Y, T)).astype(np.float32))
    net = FnoGpu(cfg, p)
    assert net.fused
    plain, saved, grads = {}, {}, {}
    for fused in (True, False):
        net.fused = fused
        plain[fused] = net.forward(dx).numpy().astype(np.float64)
        y = net.forward(dx, keep=True).numpy()
        st = net._st
        saved[fused] = {"y": y, **{n: st[n].numpy() for n in ("v1", "z0", "v2", "z1", "V30", "V32", "vL")}}
        loss = net.loss_and_grad(dx, tgt)
        grads[fused] = {"loss": np.float64(loss), **net.grads()}
    for n, b in saved[False].items():
        assert np.array_equal(saved[True][n], b), n
    assert np.linalg.norm(plain[True] - plain[False]) <= 1e-4 * np.linalg.norm(plain[False] - x[:, :2])
    assert abs(grads[True]["loss"] - grads[False]["loss"]) <= 1e-6 * grads[False]["loss"]
    for n, b in grads[False].items():
        a = grads[True][n]
        if n[0] == "R":
            assert np.array_equal(a, b), n
        else:
            assert np.abs(a - b).max() <= 1e-4 * np.abs(b).max(), n


@pytest.mark.parametrize("B,no,ni,npts", [(3, 32, 32, 120044), (3, 64, 64, 120044), (2, 33, 17, 300004),
                                          (5, 2, 4, 70012)])
def test_weight_gradients_over_several_rounds(gpu_lib, B, no, ni, npts):
    """dW += sum d x^T and db = sum d against float64 on operands rounded to BF16
    (d in full for db), a workgroup taking r chunks of 256 points, some from one
    sample and some from the next, the last of a sample ragged.  A sum passes
    through at most 64 r additions in a wave, 3 over the waves, 16 + 32 over the
    workgroups and one to dW: within that many times 2^-24 of the sum of the
    terms' magnitudes"""
    import torch
    from mpc_amd.fno import DArr, Ops
    chunks = B * -(-npts // 256)
    rounds = -(-chunks // 512)
    print(f"case wgrad rounds B={B} no={no} ni={ni} np={npts} rounds={rounds}", flush=True)
    assert rounds >= 3 and npts % 256
    rng = np.random.default_rng(npts)
    d, x = (rng.standard_normal((B, n, npts)).astype(np.float32) for n in (no, ni))
    w0 = rng.standard_normal((no, ni)).astype(np.float32)
    o, dW, db = Ops(), DArr.of(w0), DArr((no,)).fill(9.0)
    assert 0 < gpu_lib.mpc_fno_wgrad_ws(no, ni, npts) <= 4 * o.ws.numel()
    o.wgrad(DArr.of(d), DArr.of(x), dW, db, no, ni, npts, B)
    rd, rx = (torch.from_numpy(a).to(torch.bfloat16).double().numpy() for a in (d, x))
    tol = (64 * rounds + 3 + 16 + 32 + 1) * 2.0 ** -24
    ref = sum(rd[b] @ rx[b].T for b in range(B))
    mag = sum(np.abs(rd[b]) @ np.abs(rx[b]).T for b in range(B))
    assert (np.abs(dW.numpy() - (w0 + ref)) <= tol * (mag + np.abs(w0))).all()
    d = d.astype(np.float64)
    assert (np.abs(db.numpy() - d.sum((0, 2))) <= tol * np.abs(d).sum((0, 2))).all()


@pytest.mark.parametrize("nslice,m,kk,nq,h", [(3, 8, 65, 2, 7), (5, 17, 100, 1, 32), (2, 64, 128, 3, 33),
                                              (4, 33, 96, 1, 16), (3, 50, 31, 4, 9)])
@pytest.mark.parametrize("bwd", [False, True])
def test_dft_past_64_matches_separate_kernels(gpu_lib, nslice, m, kk, nq, h, bwd):
    """the truncated DFT and its transpose where the contraction (kk, 2 m) takes
    five to eight steps of 16, against the GEMM and the recombination: the same
    operands, roundings and order, the same bits"""
    from mpc_amd.fno import DArr, Ops
    print(f"case dft nslice={nslice} m={m} kk={kk} nq={nq} h={h} bwd={bwd}", flush=True)
    assert gpu_lib.mpc_fno_dft_fits(m, kk, bwd)
    rng = np.random.default_rng(m + kk)
    row = nq * 2 * h
    G = DArr.of(rng.standard_normal((2 * m, kk)))
    src = DArr.of(rng.standard_normal((nslice, m if bwd else kk, row)))
    o, got, ref = Ops(), DArr((nslice, kk if bwd else m, row)), DArr((nslice, kk if bwd else m, row))
    P = DArr((nslice, 2 * m, row))
    for sign in (-1, 1):
        o.dft(o.pack(G, 1 if bwd else 0, m, kk), src, got, nslice, m, kk, nq, h, sign, bwd=bwd)
        if bwd:
            o.combine(src, P, nslice, m, nq, h, sign, bwd=True)
            o.gemm(kk, row, 2 * m, G, 1, kk, P, row, 1, ref, row, 1, b1=(nslice, 0, 2 * m * row, kk * row))
        else:
            o.gemm(2 * m, row, kk, G, kk, 1, src, row, 1, P, row, 1, b1=(nslice, 0, kk * row, 2 * m * row))
            o.combine(P, ref, nslice, m, nq, h, sign)
        assert np.array_equal(got.numpy(), ref.numpy())
