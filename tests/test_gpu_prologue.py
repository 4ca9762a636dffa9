"""Fused camera + RMSNorm + RoPE prologue against the fp32/f64 oracle."""

import numpy as np
import pytest
import torch

from multics_amd.kernels import qkv_prologue
from oracle import attention as OA
from tests.gpu_util import err_stats, need_gpu, say

pytestmark = pytest.mark.gpu


def _freqs(P, T, h, w, KG_total):
    bands = OA.rerope_bands(128)
    verts = OA.simplex_vertices(10, 32)
    agent = torch.cat([OA.player_freqs(bands, T, h, w, verts, p) for p in range(P)], 0)
    return torch.cat([agent, OA.hub_freqs(bands, T, KG_total)], 0)


@pytest.mark.parametrize("camera", [False, True])
@pytest.mark.parametrize("layout", ["shd", "hsd"])
@pytest.mark.parametrize("shape", ["small", "odd_tokens", "dim4096", "dim3072", "dim768", "d64"])
def test_prologue_matches_oracle(camera, layout, shape):
    """Model dims that are multiples of 512 run one wave per token run
    (row_prologue_kernel), others the workgroup-per-token kernel.  small: 168
    tokens, dim 512; odd_tokens: 141 tokens, so a wave's run ends on a token
    paired with itself; dim4096: 32 heads (eight chunks per lane); dim3072:
    the C2 model dim (six chunks), with camera rows changing inside a wave's
    run; dim768: 6 heads, the workgroup kernel; d64: head dim 64, 8 heads
    (dim 512, the wave kernel's D = 64 pair indexing)."""
    need_gpu()
    say("prologue camera", camera, layout, shape)
    P, T, h, w, H, D = 2, 3, 4, 5, 4, 128
    if shape == "d64":
        H, D = 8, 64
    K_total = 2 * 5 + 6
    if shape == "odd_tokens":
        h, w, K_total = 3, 5, 2 * 5 + 7
    elif shape == "dim4096":
        T, H = 2, 32
    elif shape == "dim3072":
        T, H = 2, 24
    elif shape == "dim768":
        H = 6
    S = P * T * h * w + T * K_total
    assert shape != "odd_tokens" or S % 2 == 1
    dim = H * D
    g = torch.Generator().manual_seed(5)
    qx = (torch.randn(S, dim, generator=g) * 0.7).to(torch.bfloat16)
    kx = (torch.randn(S, dim, generator=g) * 0.7).to(torch.bfloat16)
    vx = torch.randn(S, dim, generator=g).to(torch.bfloat16)
    wq = (1 + 0.1 * torch.randn(dim, generator=g)).to(torch.bfloat16)
    wk = (1 + 0.1 * torch.randn(dim, generator=g)).to(torch.bfloat16)
    freqs = _freqs(P, T, h, w, K_total)
    if D == 64:
        freqs = freqs[..., :32].contiguous()   # any unit rotations serve the comparison
    cam = wcq = wck = None
    if camera:
        cam = torch.zeros(S, 12)
        cam[:P * T * h * w] = torch.randn(P * T * h * w, 12, generator=g)
        cam = cam.to(torch.bfloat16)
        wcq = (0.05 * torch.randn(dim, 12, generator=g)).to(torch.bfloat16)
        wck = (0.05 * torch.randn(dim, 12, generator=g)).to(torch.bfloat16)
    dev = "cuda"
    q, k, v = qkv_prologue(
        qx.to(dev), kx.to(dev), vx.to(dev), norm_q_w=wq.to(dev), norm_k_w=wk.to(dev),
        rope_cos=freqs[:, 0].real.float().to(dev), rope_sin=freqs[:, 0].imag.float().to(dev),
        num_heads=H, eps=1e-6, cam=None if cam is None else cam.to(dev),
        w_cam_q=None if wcq is None else wcq.to(dev), w_cam_k=None if wck is None else wck.to(dev),
        out_layout=layout)
    torch.cuda.synchronize()
    rq, rk = OA.project_qk(qx, kx, norm_q_w=wq, norm_k_w=wk, freqs=freqs, num_heads=H, eps=1e-6,
                           cam=cam, w_cam_q=wcq, w_cam_k=wck)
    for got, ref in ((q, rq), (k, rk)):
        got = got.reshape(S, dim)
        mx, mn = err_stats(got, ref)
        same = (got.float().cpu() == ref).float().mean().item()
        say(f"  max-abs {mx:.3e} mean-abs {mn:.3e} identical {same:.5f}")
        assert mx <= 2e-2 and mn <= 2e-4 and same > 0.99
    assert torch.equal(v.reshape(S, dim).cpu(), vx)


def test_prologue_c2_full_size():
    """The prologue exactly as ``bench.py`` times it: C2 (37,632 tokens x
    3,072 channels, 24 heads), camera12 of the bench's seeded poses, the
    bench's fp32 simplex RoPE table, head-major output.  Each output token
    depends only on its own row, so sampled tokens are compared with
    ``project_qk`` over an f64 RoPE table built by the oracle: the first and
    last token of every (player, frame) camera run, every hub row of the
    first, middle and last frames, and random tokens."""
    need_gpu()
    import bench
    P, T, L, N, KL, KG, n, W, H, D, _ = bench.CONFIGS["c2"]
    K = N * KL + KG
    S, dim = P * T * L + T * K, H * D
    dev = "cuda"
    say("prologue c2 full size", S, dim)
    g = torch.Generator(device=dev).manual_seed(bench.SEED + 7)
    qx = (torch.randn(S, dim, generator=g, device=dev) * 0.5).to(torch.bfloat16)
    kx = (torch.randn(S, dim, generator=g, device=dev) * 0.5).to(torch.bfloat16)
    wq = (1 + 0.1 * torch.randn(dim, generator=g, device=dev)).to(torch.bfloat16)
    wk = (1 + 0.1 * torch.randn(dim, generator=g, device=dev)).to(torch.bfloat16)
    wcq = (0.02 * torch.randn(dim, 12, generator=g, device=dev)).to(torch.bfloat16)
    wck = (0.02 * torch.randn(dim, 12, generator=g, device=dev)).to(torch.bfloat16)
    cam = bench.camera_tokens(P, T, L, K, dev)
    cos, sin = bench.rope_tables(P, T, L, K, D, dev)
    q, k, _ = qkv_prologue(qx, kx, None, norm_q_w=wq, norm_k_w=wk, rope_cos=cos, rope_sin=sin,
                           num_heads=H, eps=1e-6, cam=cam, w_cam_q=wcq, w_cam_k=wck,
                           out_layout="hsd")
    torch.cuda.synchronize()
    rng = np.random.default_rng(3)
    rows = set(rng.choice(S, 1500, replace=False).tolist())
    for p in range(P):
        for t in range(T):
            base = p * T * L + t * L
            rows |= {base, base + L - 1}
    for t in (0, T // 2, T - 1):
        rows |= {P * T * L + t * N * KL + i for i in range(N * KL)}
        rows |= {P * T * L + T * N * KL + t * KG + i for i in range(KG)}
    rows = torch.tensor(sorted(rows))
    bands = OA.rerope_bands(D)
    verts = OA.simplex_vertices(10, 32)
    h, w = 11, 20
    freqs = torch.cat([OA.player_freqs(bands, T, h, w, verts, p) for p in range(P)]
                      + [OA.hub_freqs(bands, T, K)], 0)
    assert freqs.shape[0] == S
    cpu = lambda t: t.cpu()
    rq, rk = OA.project_qk(cpu(qx)[rows], cpu(kx)[rows], norm_q_w=cpu(wq), norm_k_w=cpu(wk),
                           freqs=freqs[rows], num_heads=H, eps=1e-6, cam=cpu(cam)[rows],
                           w_cam_q=cpu(wcq), w_cam_k=cpu(wck))
    for got, ref in ((q, rq), (k, rk)):
        got = got[rows.to(dev)].reshape(len(rows), dim)
        mx, mn = err_stats(got, ref)
        same = (got.float().cpu() == ref).float().mean().item()
        say(f"  {len(rows)} tokens: max-abs {mx:.3e} mean-abs {mn:.3e} identical {same:.5f}")
        assert mx <= 2e-2 and mn <= 2e-3 and same > 0.99


def _grad_check(name, got, ref, rel_max=2e-2, rel_mean=1e-2, absolute=True):
    """Relative bounds (max error within 2 % of max|ref|, mean error within
    1 % of mean|ref|) and, with ``absolute``, the north-star absolute bounds
    scaled to the gradient's size (max-abs <= 2e-2 and mean-abs <= 2e-3 per
    unit of max|ref| above 1)."""
    got = got.detach().float().cpu()
    ref = ref.detach().float()
    err = (got - ref).abs()
    scale = max(1.0, ref.abs().max().item())
    say(f"  {name}: max-abs {err.max().item():.3e} mean-abs {err.mean().item():.3e} "
        f"(ref max {ref.abs().max().item():.3e} mean {ref.abs().mean().item():.3e})")
    assert torch.isfinite(got).all(), name
    if absolute:
        assert err.max().item() <= 2e-2 * scale and err.mean().item() <= 2e-3 * scale, name
    assert err.max().item() <= rel_max * ref.abs().max().item() + 1e-6, name
    assert err.mean().item() <= rel_mean * ref.abs().mean().item() + 1e-7, name


@pytest.mark.parametrize("camera", [False, True])
@pytest.mark.parametrize("shape", ["dim512", "dim3072", "d64"])
def test_prologue_backward_matches_fp32_autograd(camera, shape):
    """``QKPrologueFunction`` (HIP forward and backward of the camera add,
    RMSNorm, gain and RoPE) against torch autograd through ``project_qk`` in
    fp32 / f64 on the CPU (the roundings of the forward pass the gradient
    through unchanged in both): gradients of the q / k projections, the
    RMSNorm gains and the camera-adapter weights."""
    need_gpu()
    from multics_amd.kernels import qk_prologue_train
    say("prologue backward", shape, "camera", camera)
    P, T, h, w, H, D = 2, 3, 4, 5, 4, 128
    if shape == "dim3072":
        T, H = 2, 24
    elif shape == "d64":
        H, D = 8, 64
    K_total = 2 * 5 + 6
    S = P * T * h * w + T * K_total
    dim = H * D
    g = torch.Generator().manual_seed(8)
    qx = (torch.randn(S, dim, generator=g) * 0.5).to(torch.bfloat16)
    kx = (torch.randn(S, dim, generator=g) * 0.5).to(torch.bfloat16)
    wq = (1 + 0.1 * torch.randn(dim, generator=g)).to(torch.bfloat16)
    wk = (1 + 0.1 * torch.randn(dim, generator=g)).to(torch.bfloat16)
    freqs = _freqs(P, T, h, w, K_total)
    if D == 64:
        freqs = freqs[..., :32].contiguous()
    cam = wcq = wck = None
    if camera:
        cam = torch.zeros(S, 12)
        cam[:P * T * h * w] = torch.randn(P * T * h * w, 12, generator=g)
        cam = cam.to(torch.bfloat16)
        wcq = (0.05 * torch.randn(dim, 12, generator=g)).to(torch.bfloat16)
        wck = (0.05 * torch.randn(dim, 12, generator=g)).to(torch.bfloat16)
    dq = (torch.randn(S, H, D, generator=g) * 0.5).to(torch.bfloat16)
    dk = (torch.randn(S, H, D, generator=g) * 0.5).to(torch.bfloat16)

    dev = "cuda"
    leaf = lambda t: None if t is None else t.to(dev).requires_grad_(True)
    hq, hk, hwq, hwk, hwcq, hwck = (leaf(t) for t in (qx, kx, wq, wk, wcq, wck))
    q, k = qk_prologue_train(hq, hk, norm_q_w=hwq, norm_k_w=hwk,
                             rope_cos=freqs[:, 0].real.float().to(dev),
                             rope_sin=freqs[:, 0].imag.float().to(dev), num_heads=H, eps=1e-6,
                             cam=None if cam is None else cam.to(dev), w_cam_q=hwcq, w_cam_k=hwck)
    torch.autograd.backward([q, k], [dq.to(dev), dk.to(dev)])
    torch.cuda.synchronize()

    f32 = lambda t: None if t is None else t.float().requires_grad_(True)
    rq, rk, rwq, rwk, rwcq, rwck = (f32(t) for t in (qx, kx, wq, wk, wcq, wck))
    oq, ok = OA.project_qk(rq, rk, norm_q_w=rwq, norm_k_w=rwk, freqs=freqs, num_heads=H, eps=1e-6,
                           cam=None if cam is None else cam.float(), w_cam_q=rwcq, w_cam_k=rwck)
    torch.autograd.backward([oq, ok], [dq.float().reshape(S, dim), dk.float().reshape(S, dim)])
    for name, a, b in (("dqx", hq.grad, rq.grad), ("dkx", hk.grad, rk.grad),
                       ("dnorm_q", hwq.grad, rwq.grad), ("dnorm_k", hwk.grad, rwk.grad)):
        _grad_check(name, a, b)
    if camera:
        _grad_check("dcam_q", hwcq.grad, rwcq.grad)
        _grad_check("dcam_k", hwck.grad, rwck.grad)


@pytest.mark.parametrize("S,H,D,run", [
    (1, 4, 128, 1),          # one token, one workgroup, three of its four padded rows empty
    (8, 8, 64, 3),           # exactly one workgroup of 8 tokens, a camera row change inside a trip
    (13, 8, 128, 1),         # every token its own camera row; a last trip of one token
    (1030, 12, 128, 37),     # workgroups of 8 tokens, camera runs that cross them
    (1100, 24, 128, 220),    # 9 tokens per workgroup: a ragged last trip in each
    (70, 28, 128, 5),        # 8 channels per thread, two tokens per trip, odd runs
    (70, 64, 64, 70),        # the largest model dim
    (1536, 24, 128, 1),      # 12 tokens and camera rows per workgroup: its slots just hold them
    (1664, 24, 128, 1),      # 13: the row past the slots is the last token's
    (1700, 24, 128, 1),      # 14: one row more, and a last workgroup of 6
    (3200, 24, 128, 1),      # 25: as many rows again after the slots are full
    (3200, 24, 128, 2),      # 13 rows of two tokens, runs that cross workgroups
])
def test_prologue_backward_sums(S, H, D, run):
    """The sums over tokens of the prologue backward (gain and camera-weight
    gradients) and the projections' gradients, where the token split, the
    trips and the camera runs (``run`` tokens of one row, every third run
    zeros) can go wrong, against float64 autograd.  Bounds: results are bf16
    (2^-8 of the value) of fp32 sums of terms with the forward's bf16 rounding
    of a (2^-8 of each term): 1 % of the largest entry."""
    need_gpu()
    from multics_amd.kernels import qk_prologue_train
    say("prologue backward sums", S, H, D, run)
    dim = H * D
    g = torch.Generator().manual_seed(S + H)
    bf = lambda *s, std=1.0: (std * torch.randn(*s, generator=g)).to(torch.bfloat16)
    qx, kx = bf(S, dim), bf(S, dim)
    wq, wk = (1 + 0.1 * torch.randn(2, dim, generator=g)).to(torch.bfloat16)
    wcq, wck = bf(dim, 12, std=0.05), bf(dim, 12, std=0.05)
    rows = bf(-(-S // run), 12)
    rows[2::3] = 0
    cam = rows.repeat_interleave(run, 0)[:S].contiguous()
    ang = 6.283 * torch.rand(S, D // 2, generator=g, dtype=torch.float64)
    cos, sin = ang.cos(), ang.sin()
    dq, dk = bf(S, H, D), bf(S, H, D)
    leaf = lambda t: t.cuda().requires_grad_(True)
    hip = [leaf(t) for t in (qx, kx, wq, wk, wcq, wck)]
    q, k = qk_prologue_train(hip[0], hip[1], norm_q_w=hip[2], norm_k_w=hip[3],
                             rope_cos=cos.float().cuda(), rope_sin=sin.float().cuda(), num_heads=H,
                             eps=1e-6, cam=cam.cuda(), w_cam_q=hip[4], w_cam_k=hip[5])
    got = torch.autograd.grad((q, k), hip, (dq.cuda(), dk.cuda()))
    torch.cuda.synchronize()

    ref = [t.double().requires_grad_(True) for t in (qx, kx, wq, wk, wcq, wck)]

    def tail(x, w, wc):
        a = x + cam.double() @ wc.t()
        z = (a * torch.rsqrt(a.square().mean(-1, keepdim=True) + 1e-6) * w).view(S, H, D // 2, 2)
        c, s = cos[:, None], sin[:, None]
        return torch.stack([z[..., 0] * c - z[..., 1] * s, z[..., 0] * s + z[..., 1] * c],
                           -1).flatten(2)

    want = torch.autograd.grad((tail(ref[0], ref[2], ref[4]), tail(ref[1], ref[3], ref[5])), ref,
                               (dq.double(), dk.double()))
    for name, a, b in zip(("dqx", "dkx", "dnorm_q", "dnorm_k", "dcam_q", "dcam_k"), got, want):
        err = (a.double().cpu() - b).abs().max().item()
        say(f"  {name}: max-abs {err:.3e} of {b.abs().max().item():.3e}")
        assert err <= 1e-2 * b.abs().max().item(), name


def _tail_inputs(S, H, D, seed):
    g = torch.Generator().manual_seed(seed)
    bf = lambda *s, std=1.0: (std * torch.randn(*s, generator=g)).to("cuda", torch.bfloat16)
    dim = H * D
    ang = 6.283 * torch.rand(S, D // 2, generator=g).cuda()
    return dict(qx=bf(S, dim), kx=bf(S, dim), norm_q_w=1 + bf(dim, std=0.1),
                norm_k_w=1 + bf(dim, std=0.1), cam=bf(S, 12), w_cam_q=bf(dim, 12, std=0.05),
                w_cam_k=bf(dim, 12, std=0.05), cos=ang.cos(), sin=ang.sin(), dq=bf(S, H, D),
                dk=bf(S, H, D))


@pytest.mark.parametrize("frozen", ["both", "q", "k"])
def test_prologue_backward_with_frozen_camera_weights(frozen):
    """Camera weights that take no gradient change nothing in the others' (with
    both frozen the pass keeps no camera sums)."""
    need_gpu()
    from multics_amd.kernels import qk_prologue_train
    say("prologue backward, frozen camera weights", frozen)
    S, H, D = 100, 4, 128
    t = _tail_inputs(S, H, D, 5)
    names = ["qx", "kx", "norm_q_w", "norm_k_w", "w_cam_q", "w_cam_k"]

    def grads(off):
        x = {n: t[n].clone().requires_grad_(n not in off) for n in names}
        q, k = qk_prologue_train(x["qx"], x["kx"], norm_q_w=x["norm_q_w"], norm_k_w=x["norm_k_w"],
                                 rope_cos=t["cos"], rope_sin=t["sin"], num_heads=H, eps=1e-6,
                                 cam=t["cam"], w_cam_q=x["w_cam_q"], w_cam_k=x["w_cam_k"])
        torch.autograd.backward([q, k], [t["dq"], t["dk"]])
        return {n: x[n].grad for n in names}

    off = {"both": {"w_cam_q", "w_cam_k"}, "q": {"w_cam_q"}, "k": {"w_cam_k"}}[frozen]
    want, got = grads(set()), grads(off)
    for n in names:
        if n in off:
            assert got[n] is None
        else:
            assert torch.equal(got[n], want[n]), n


@pytest.mark.parametrize("S,H,D,tokens", [(1, 4, 128, 16), (37, 24, 128, 5), (1000, 8, 64, 16),
                                          (130, 64, 64, 33)])
def test_prologue_backward_partial_rows(S, H, D, tokens):
    """``hier_qk_prologue_bwd``, whose caller adds the partial rows itself: the
    projections' gradients are those of ``hier_qk_prologue_grads``, and the
    rows' sums are its gain gradients before their rounding to bf16 (2^-8 of
    the value, half a unit of 8 bits, and fp32 sums in another order)."""
    need_gpu()
    import ctypes as C

    from multics_amd import _capi
    say("prologue backward partial rows", S, H, D, tokens)
    dim = H * D
    t = _tail_inputs(S, H, D, 6)
    new = lambda *s, dtype=torch.bfloat16: torch.full(s, float("nan"), dtype=dtype, device="cuda")
    stream = _capi.stream_of(t["qx"].device)

    def run(grads):
        dqx, dkx = new(S, dim), new(S, dim)
        a = _capi.HierPrologueBwdArgs(
            S=S, H=H, D=D, eps=1e-6, C=12, tokens_per_wave=tokens, qx=t["qx"].data_ptr(),
            kx=t["kx"].data_ptr(), cam=t["cam"].data_ptr(), w_cam_q=t["w_cam_q"].data_ptr(),
            w_cam_k=t["w_cam_k"].data_ptr(), norm_q_w=t["norm_q_w"].data_ptr(),
            norm_k_w=t["norm_k_w"].data_ptr(), rope_cos=t["cos"].data_ptr(),
            rope_sin=t["sin"].data_ptr(), dq=t["dq"].data_ptr(), dk=t["dk"].data_ptr(), dq_ss=dim,
            dq_sh=D, dk_ss=dim, dk_sh=D, dqx=dqx.data_ptr(), dkx=dkx.data_ptr())
        rows = _capi.lib().hier_qk_prologue_bwd_waves(C.byref(a))
        assert rows >= -(-S // tokens)
        part = new(2, rows, dim, dtype=torch.float32)
        a.dw_q_partial, a.dw_k_partial = part[0].data_ptr(), part[1].data_ptr()
        dn = new(2, dim)
        if grads:
            g = _capi.HierPrologueGradArgs(dnorm_q=dn[0].data_ptr(), dnorm_k=dn[1].data_ptr())
            _capi.call("hier_qk_prologue_grads", C.byref(a), C.byref(g), stream)
        else:
            _capi.call("hier_qk_prologue_bwd", C.byref(a), stream)
        torch.cuda.synchronize()
        return dqx, dkx, part.double().sum(1), dn.double()

    dqx, dkx, sums, _ = run(False)
    dqx2, dkx2, _, dn = run(True)
    assert torch.equal(dqx, dqx2) and torch.equal(dkx, dkx2)
    assert not dqx.isnan().any() and not sums.isnan().any()
    assert ((dn - sums).abs() <= 2.0 ** -8 * sums.abs() + 1e-5 * sums.abs().max()).all()
