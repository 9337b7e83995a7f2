"""GPU: the GEMM path (more than 64 rows; 33-64 rows whose latent vectors do not
fit the decode path's buffer) at the edges of its tiles, its k parts and its
sign-word loads, in its split (fp32) and bf16 forms, against the oracle."""
import numpy as np
import pytest
import torch

import oracle.littlebit_oracle as O

pytestmark = pytest.mark.gpu

# hi + lo planes keep 16-17 mantissa bits of every product's activation
# (2**-17 of its magnitude, in each stage), as on the decode path: the largest
# difference over the largest result measures 3.5e-6, a few standard deviations
# of the sums' error are 4e-5, and a branch without its lo plane shows 5.8e-4
# (A's) or 6.8e-4 (T's).  bf16 calls round x * g (or g) and the latent vector to
# 2**-9 of their magnitudes.
TOL = {torch.float32: 4e-5, torch.bfloat16: 5e-3}


def _make(gpu, seed, M, K, specs, x_dtype, tile_v=True, offset=0):
    from littlebit_amd import LittleBitBranch, LittleBitProjection, LittleBitProjectionGroup
    from littlebit_amd.synthetic import make_branch
    rng = np.random.Generator(np.random.PCG64(seed))
    host = [[make_branch(rng, K, R, N) for R in ranks] for N, ranks in specs]
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)  # noqa: E731
    projs = [LittleBitProjection([LittleBitBranch(t(b.v_sign), t(b.u_sign), t(b.g), t(b.l), t(b.h)) for b in brs],
                                 tile_v=tile_v) for brs in host]
    buf = torch.zeros(M * K + offset, dtype=x_dtype, device=gpu)
    x = buf[offset:].view(M, K)
    x.copy_(torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).to(gpu))
    return host, LittleBitProjectionGroup(projs), x


def _check(host, specs, K, x, outs, rows=None, tol=TOL[torch.float32]):
    xu = x.float().cpu().numpy()
    rows = np.arange(xu.shape[0]) if rows is None else rows
    for (N, _), brs, y in zip(specs, host, outs):
        ref = O.littlebit_forward(xu[rows], [b.as_dict() for b in brs], K, N)
        err = O.rel_err(y.cpu().numpy()[rows], ref)
        print(f"[split] M={xu.shape[0]} K={K} N={N} rel_err={err:.2e}", flush=True)
        assert err <= tol, (N, err)


@pytest.mark.parametrize("x_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,K,specs", [
    (65, 4096, [(4096, [205, 1843])]),              # k in parts, one row past two row tiles
    (97, 1000, [(300, [127, 129])]),                # K off the word groups, ranks at a group's edge
    (70, 33, [(1, [1, 5])]),                        # sign matrices of fewer than 4 words
    (66, 32, [(3, [32]), (2, [70, 3])]),            # one-word rows, two projections
    (128, 130, [(129, [128, 96]), (257, [31])]),    # last word partly used; one and two branches
    (200, 260, [(4500, [40, 600])]),                # stage 2: 245 tiles of 32 x 128, ranks past 16 steps
    (1100, 200, [(5000, [40, 600])]),               # stage 2 as 64 x 128 tiles, partial last tiles
    (1100, 200, [(9000, [40, 601])]),               # stage 2 as 64 x 256 tiles, partial last tiles
    (2049, 264, [(130, [205, 3000])]),              # stage 1 as 64-row tiles
    (2049, 320, [(130, [205, 3000])]),              # the same, bf16 rows read as they are, an odd step
    (330, 8256, [(130, [205, 1843])]),              # long rows: 64-row tiles in parts
    (2049, 8384, [(130, [40, 2900])]),              # long rows, bf16 as 128-row tiles: three steps past the ring's rounds
    (2049, 8200, [(130, [40, 2900])]),              # the same from a scaled copy (K off the steps)
])
def test_sign_gemm_edges(gpu, M, K, specs, x_dtype):
    """(Which kernels these shapes run is checked in tests/sanitize/abi_host_check.cpp.)"""
    host, grp, x = _make(gpu, 9100 + M, M, K, specs, x_dtype)
    a = grp.forward(x, out_dtype=torch.float32)
    b = grp.forward(x, out_dtype=torch.float32)
    torch.cuda.synchronize()
    rows = np.unique(np.r_[0:min(M, 40), max(0, M - 70):M])  # rows are independent
    _check(host, specs, K, x, a, rows, TOL[x_dtype])
    for u, v in zip(a, b):
        assert torch.equal(u, v), "the GEMM path repeats bit for bit"
    host2, stored, x2 = _make(gpu, 9100 + M, M, K, specs, x_dtype, tile_v=False)
    for u, v in zip(a, stored.forward(x2, out_dtype=torch.float32)):
        assert torch.equal(u, v), "V as stored and V tiled hold the same signs"


@pytest.mark.parametrize("M,x_dtype,offset", [(64, torch.float32, 0), (47, torch.bfloat16, 0), (100, torch.float32, 1)])
def test_sign_gemm_inputs(gpu, M, x_dtype, offset):
    """RMSNorm, SiLU * up and plain inputs, residual in place, rows that take
    the path because their latent vectors do not fit the decode buffer (two
    projections of ranks 298 + 2686: 46 rows do not), misaligned x."""
    K, specs = 520, [(1030, [298, 2686]), (514, [298, 2686])]
    host, grp, x = _make(gpu, 9300 + M, M, K, specs, x_dtype, offset=offset)
    gen = torch.Generator(device=gpu).manual_seed(M)
    w = 1 + 0.1 * torch.randn(K, generator=gen, device=gpu)
    up = torch.randn((M, K), generator=gen, device=gpu).to(x_dtype)
    outs = [torch.randn((M, N), generator=gen, device=gpu) for N, _ in specs]
    before = [o.clone() for o in outs]
    grp.forward(x, outs=outs, out_dtype=torch.float32, residuals=outs, rms_weight=w)
    xd = x.double()
    h = (xd / torch.sqrt((xd * xd).mean(-1, keepdim=True) + 1e-6) * w.double()).float()
    _check(host, specs, K, h, [o - r for o, r in zip(outs, before)])
    outs = grp.forward(x, out_dtype=torch.float32, x_up=up)
    _check(host, specs, K, (xd / (1 + torch.exp(-xd)) * up.double()).float(), outs)
    _check(host, specs, K, x, grp.forward(x, out_dtype=torch.float32))


@pytest.mark.parametrize("M,N,ranks", [
    (72, 176, [64, 200]),     # stage 2 as 32 x 128 tiles
    (1100, 5000, [40, 600]),  # 64 x 128
    (1100, 9000, [601, 40]),  # 64 x 256
])
def test_sign_gemm_scale_ratios(gpu, M, N, ranks):
    """Both branches share one accumulator set, rescaled by the ratio of
    their row scales between them: ratios up to 2**+-60 with sums as large as
    their product with the ratio still representable, zeros, and infinities
    and NaN in either scale give what the formula has."""
    K = 256
    host, grp, x = _make(gpu, 9500, M, K, [(N, ranks)], torch.float32)
    brs = host[0]
    h0, h1 = brs[0].h, brs[1].h
    for i in range(0, 120, 2):
        h1[i] = h0[i] * np.float32(2.0 ** -(i // 2))
        h0[i + 1] = h1[i + 1] * np.float32(2.0 ** -(i // 2))
    h1[120:130] = 0.0
    h0[130:140] = 0.0
    h0[160:162] = np.inf
    h1[162:164] = -np.inf
    h0[164:166] = np.nan
    h1[166:168] = np.nan
    h0[168], h1[168] = -np.inf, 0.0
    finite = np.r_[0:160, 169:N]
    big = np.float32(1e25)
    grp.projections[0].branches[0].u1.copy_(torch.from_numpy(h0))
    grp.projections[0].branches[1].u1.copy_(torch.from_numpy(h1))
    rows = np.unique(np.r_[0:40, M - 40:M])  # rows are independent
    for scale in (np.float32(1), big):
        xs = x * float(scale)
        y = grp.forward(xs)[0].cpu().numpy().astype(np.float64)[rows]
        with np.errstate(invalid="ignore"):
            ref = O.littlebit_forward(xs.cpu().numpy()[rows], [b.as_dict() for b in brs], K, N)
        # per column: each column has its own scale
        err = np.abs(y - ref)[:, finite].max(0) / np.abs(ref[:, finite]).max(0)
        print(f"[split] M={M} ratios scale={scale:g} worst column {err.max():.2e}", flush=True)
        assert np.isfinite(y[:, finite]).all() and err.max() <= TOL[torch.float32]
        assert np.array_equal(y[:, 160:169], ref[:, 160:169], equal_nan=True)
        assert np.isinf(y[:, 160:164]).all() and np.isnan(y[:, 164:168]).all()


@pytest.mark.parametrize("M", [70, 300, 1024])
def test_two_branches_are_as_exact_as_a_call_each(gpu, M):
    """Both branches of a call share one set of sums in stage 2.  The branch
    of the smaller rank comes second, whatever order the caller has them in:
    its 7 words' 28 MFMAs and the rescale round at the size of the whole sum,
    sqrt(30) * 2**-24 / sqrt(3) = 1.9e-7 of it at most beside 3.5e-6 from the
    planes, 0.15 % in quadrature (1,843 columns second: 0.3 to 0.6 %)."""
    from littlebit_amd import LittleBitProjection
    K, N, ranks = 4096, 4096, [205, 1843]
    joined, apart = [], []
    for seed in (9700, 9701):
        _, grp, x = _make(gpu, seed, M, K, [(N, ranks)], torch.float32)
        brs = grp.projections[0].branches
        for b, r in zip(brs, ranks):
            b.mid.div_(r ** 0.5)  # branches of equal size, as in a trained model
        pm1 = lambda w, n: (1 - 2 * ((w.unsqueeze(-1) >> torch.arange(32, dtype=torch.int32, device=gpu)) & 1)  # noqa: E731
                            ).reshape(w.shape[0], -1)[:, :n].double()
        ref = sum(((x.double() * b.v2.double()) @ pm1(b.v_sign, K).t().contiguous() * b.mid.double())
                  @ pm1(b.u_sign, b.mid.numel()).t().contiguous() * b.u1.double() for b in brs)
        err = lambda y: float((y.double() - ref).norm() / ref.norm())  # noqa: E731
        y = LittleBitProjection(brs).forward(x)
        assert torch.equal(y, LittleBitProjection(brs[::-1]).forward(x)), "the caller's order changes nothing"
        joined.append(err(y))
        apart.append(err(sum(LittleBitProjection([b]).forward(x) for b in brs)))
    print(f"[split] M={M} joined {joined} apart {apart}", flush=True)
    assert sum(joined) <= 1.002 * sum(apart)
