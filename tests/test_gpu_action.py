"""Action branches' cached attention on the GPU: the frame-window attention
kernel against the oracle's masked SDPA, and the mouse temporal /
keyboard cached attention over a rollout (every block run twice) against the
full-sequence computation with the same mask, which an in-order rollout
equals.  Bound: max-abs 2e-2, mean-abs 2e-3 against fp32."""

import copy
import math

import pytest
import torch
from torch import nn

from multics_amd.action import (
    action_keyboard_cached_attention,
    action_temporal_cached_attention,
    frame_attention,
)
from multics_amd.rope import precompute_freqs_cis
from oracle.cached import _sdpa, _temporal
from tests.gpu_util import err_stats, need_gpu, say

pytestmark = pytest.mark.gpu
MAX_ABS, MEAN_ABS = 2e-2, 2e-3


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("local_attn", [-1, 5])
def test_frame_attention_matches_oracle(D, local_attn):
    need_gpu()
    say("frame attention", D, local_attn)
    g = torch.Generator().manual_seed(D + local_attn)
    B, H, n_block = 5, 3, 3
    for Lq, Lk, q0 in ((3, 24, 21), (7 * 4, 9 * 2, 6), (1, 1, 0)):
        qf = q0 + torch.arange(Lq) * 3 // max(Lq, 1)        # a few frames, in order
        kf = torch.arange(Lk) * (q0 + 3) // max(Lk, 1)
        q, k, v = ((torch.randn(B, L, H, D, generator=g)).to(torch.bfloat16) for L in (Lq, Lk, Lk))
        got = frame_attention(q.cuda(), k.cuda(), v.cuda(), qf, kf, n_block, local_attn)
        torch.cuda.synchronize()
        m = _temporal(qf, kf, n_block, local_attn)
        ref = torch.stack([_sdpa(q[b], k[b], v[b], m, 1 / math.sqrt(D)) for b in range(B)])
        mx, mn = err_stats(got, ref)
        say(f"  Lq {Lq} Lk {Lk}: max-abs {mx:.3e} mean-abs {mn:.3e}")
        assert mx <= MAX_ABS and mn <= MEAN_ABS


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Lq", [1, 2, 3, 4, 5, 6, 7, 8, 9, 14, 16, 17, 32, 33, 129])
def test_frame_attention_edges(D, Lq):
    """Every kernel variant (waves of 1-8 queries, matrix tiles above) at
    the edges of its key chunks and tiles, with keys that no query, one query
    or all queries see, head counts that leave waves of a workgroup empty, and
    q / k / v as slices of larger tensors (heads before tokens for k),
    against float64.  Scores, weights and sums are fp32, so a result is off
    by its own bf16 rounding (2^-8 of it) and fp32 terms far below 1e-3 of the
    values' size."""
    need_gpu()
    g = torch.Generator().manual_seed(100 * D + Lq)
    n_block = 3
    # (a row group is 4 keys at D = 128, 8 at 64; a chunk 2, 3, 4, 6 or 8 of them)
    for B, H, Lk, W in ((3, 5, 1, -1), (1, 3, 5, 30), (2, 1, 7, -1), (1, 2, 8, 12), (1, 3, 9, 30),
                        (2, 2, 12, 21), (1, 1, 13, -1), (1, 3, 16, 30), (1, 2, 17, 12),
                        (2, 4, 24, 21), (1, 3, 25, -1), (1, 3, 31, 4), (1, 1, 32, 30),
                        (2, 2, 33, 6), (1, 2, 48, 21), (1, 1, 49, 12), (1, 1, 64, -1),
                        (2, 3, 65, 9), (1, 2, 200, 30)):
        say("frame attention edges", D, Lq, B, H, Lk, W)
        q = torch.randn(B, Lq + 2, H + 1, D, generator=g).to(torch.bfloat16)[:, 1:-1, 1:]
        k = torch.randn(B, H, Lk, D, generator=g).to(torch.bfloat16).transpose(1, 2)
        v = torch.randn(B, Lk, 2 * H, D, generator=g).to(torch.bfloat16)[:, :, :H]
        kf = torch.sort(torch.randint(0, 40, (Lk,), generator=g)).values
        qf = 12 + torch.arange(Lq) % 20
        qd, vd = (torch.zeros(t.shape[0], t.shape[1] + 2, 2 * H, D, dtype=torch.bfloat16,
                              device="cuda")[:, 1:-1, :H] for t in (q, v))
        qd.copy_(q), vd.copy_(v)
        kd = k.transpose(1, 2).contiguous().cuda().transpose(1, 2)
        got = frame_attention(qd, kd, vd, qf, kf, n_block, W)
        torch.cuda.synchronize()
        m = (kf[None] // n_block) <= (qf[:, None] // n_block)
        if W != -1:
            m &= qf[:, None] - kf[None] < W
        sc = torch.einsum("bihd,bjhd->bhij", q.double(), k.double()) / math.sqrt(D)
        p = torch.softmax(sc.masked_fill(~m, -math.inf), -1).nan_to_num(0.0)
        ref = torch.einsum("bhij,bjhd->bihd", p, v.double())
        err = (got.double().cpu() - ref).abs()
        assert (err <= 2.0 ** -8 * ref.abs() + 1e-3).all(), float(err.max())
        assert (got.cpu()[:, ~m.any(1)] == 0).all()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Lq,Lk", [(3, 24), (7, 40), (12, 70), (3, 200), (40, 96)])
def test_frame_attention_hidden_rows_count_for_nothing(D, Lq, Lk):
    """A key outside a query's window leaves that query's result alone whatever
    its K and V rows hold (infinities, NaN), in every kernel: the last row
    among them, which stands in for the rows past it, and rows that other
    queries see (whose results are then as without a mask: an infinity where V
    is infinite, NaN where a NaN takes part).  A query that sees nothing gives
    0.  Bounds as in test_frame_attention_edges."""
    need_gpu()
    say("frame attention hidden rows", D, Lq, Lk)
    g = torch.Generator().manual_seed(Lq + Lk + D)
    B, H, W = 2, 3, 6
    q, k, v = (torch.randn(B, L, H, D, generator=g).to(torch.bfloat16) for L in (Lq, Lk, Lk))
    kf = 20 + torch.arange(Lk) * 20 // Lk
    qf = torch.linspace(28, 36, Lq).long()           # frames 20-39: hidden on both sides
    qf[0] = 5                                        # sees nothing
    vis = (kf[None] <= qf[:, None]) & (qf[:, None] - kf[None] < W)
    hidden = ~vis.any(0)
    assert hidden[-1] and hidden[0]
    bad = torch.zeros(Lk, dtype=torch.bool)
    bad[-1] = bad[0] = True
    for rows, value in ((bad, float("nan")), (bad, float("inf")), (hidden, float("-inf"))):
        kk, vv = k.clone(), v.clone()
        kk[:, rows], vv[:, rows] = value, value
        # a row that only the queries of its own window see
        one = int((kf == 30).nonzero()[0])
        vv[:, one, :, 1] = float("inf")
        vv[:, one, :, 2] = float("nan")
        got = frame_attention(q.cuda(), kk.cuda(), vv.cuda(), qf, kf, 1, W).double().cpu()
        torch.cuda.synchronize()
        sc = torch.einsum("bihd,bjhd->bhij", q.double(), k.double()) / math.sqrt(D)
        p = torch.softmax(sc.masked_fill(~vis, -math.inf), -1).nan_to_num(0.0)
        ref = torch.einsum("bhij,bjhd->bihd", p, v.double())
        sees = vis[:, one]
        ref[:, sees, :, 1], ref[:, sees, :, 2] = math.inf, math.nan
        fin = torch.isfinite(ref)
        err = (got[fin] - ref[fin]).abs()
        assert (err <= 2.0 ** -8 * ref[fin].abs() + 1e-3).all(), float(err.max())
        assert (got[:, sees, :, 1] == math.inf).all() and got[:, sees, :, 2].isnan().all()
        assert (got[:, 0] == 0).all()


@pytest.mark.parametrize("Lq,Lk", [(3, 24), (3, 200), (40, 96)])
def test_frame_attention_scores_far_below_zero(Lq, Lk):
    """Scores of any finite size weigh their keys: one of -1e31 beside others
    that are lower by far takes the whole weight."""
    need_gpu()
    say("frame attention low scores", Lq, Lk)
    D = 128
    g = torch.Generator().manual_seed(Lk)
    q = torch.full((1, Lq, 2, D), 1e15).to(torch.bfloat16)
    k = torch.full((1, Lk, 2, D), -2e16).to(torch.bfloat16)
    k[:, Lk // 2] = -1e15
    v = torch.randn(1, Lk, 2, D, generator=g).to(torch.bfloat16)
    got = frame_attention(q.cuda(), k.cuda(), v.cuda(), torch.full((Lq,), 9),
                          torch.arange(Lk) % 10, 10, -1).cpu()
    torch.cuda.synchronize()
    assert torch.equal(got, v[:, Lk // 2:Lk // 2 + 1].expand_as(got))


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Lq", [3, 40])
def test_frame_attention_weights_are_fp32(D, Lq):
    """Softmax weights multiply V with all their 24 bits in every kernel.  Keys
    of weight 1, p and 1 carry v = hi, -1 and lo, the bf16 of p and the bf16
    of what that leaves: the result is what two bf16 parts of p leave out,
    over 2 + p.  Bound: the result's bf16 rounding (2^-8 of it) and the fp32
    error of p (exp2 and score, 2^-23 together)."""
    need_gpu()
    say("frame attention weights", D, Lq)
    H, scale = 48, 0.25
    x = torch.linspace(0.3, 3.0, H).to(torch.bfloat16)
    p = torch.exp(-x.double() * scale)
    hi = p.to(torch.bfloat16)
    lo = (p - hi.double()).to(torch.bfloat16)
    q, k, v = (torch.zeros(1, L, H, D, dtype=torch.bfloat16) for L in (Lq, 3, 3))
    q[..., 0] = 1
    k[0, 1, :, 0] = -x
    v[0, 0], v[0, 1], v[0, 2] = hi[:, None], -1, lo[:, None]
    got = frame_attention(q.cuda(), k.cuda(), v.cuda(), torch.zeros(Lq), torch.zeros(3), 1, -1,
                          scale=scale).double().cpu()
    torch.cuda.synchronize()
    ref = ((hi.double() - p + lo.double()) / (2 + p))[None, None, :, None].expand_as(got)
    assert (ref.abs() > 2.0 ** -21).sum() > ref.numel() / 4   # seen above the bound
    err = (got - ref).abs()
    assert (err <= 2.0 ** -8 * ref.abs() + 2.0 ** -23).all(), float(err.max())


@pytest.mark.parametrize("B,H,Lq", [(2_850_000, 24, 1), (16_800_000, 1, 17)])
def test_frame_attention_many_sequences(B, H, Lq):
    """More sequences and heads than a grid holds along x (2^26 waves; 2^24
    matrix-tile workgroups): every one is computed.  Inputs are one sequence's,
    expanded; so are its 20 keys, so the output is their V row."""
    need_gpu()
    say("frame attention many sequences", B, H, Lq)
    D = 64
    g = torch.Generator().manual_seed(H)
    q, k, v = (torch.randn(1, n, H, D, generator=g).to("cuda", torch.bfloat16).expand(B, L, H, D)
               for n, L in ((Lq, Lq), (1, 20), (1, 20)))
    got = frame_attention(q, k, v, torch.zeros(Lq), torch.zeros(20), 1, -1)
    torch.cuda.synchronize()
    step = 9973
    for part in (got[::step], got[-2:], got[B // 2:B // 2 + 2]):
        assert torch.equal(part, v[:1, :1].expand_as(part))


@pytest.mark.parametrize("B,H,Lq,Lk,D", [
    # up to 16 queries: 2 keys; at D = 64 windows of up to 4, 8 and 12 keys from
    # 2,048, 8,192 and 20,480 queries (of all sequences and heads) on; fewer
    # queries or a key more: the other kernels
    (1, 1, 1, 1, 128), (3, 5, 5, 2, 64), (2, 3, 9, 2, 128), (342, 6, 1, 4, 64), (341, 6, 1, 4, 64), (683, 6, 3, 4, 64), (683, 6, 2, 8, 64),
    (682, 6, 2, 8, 64), (683, 6, 7, 5, 64), (683, 6, 2, 9, 64), (1707, 6, 2, 12, 64),
    (1706, 6, 2, 12, 64), (1707, 6, 2, 13, 64), (214, 6, 16, 12, 64),
    # at D = 128: 4 keys from 8,192 queries on
    (683, 6, 2, 4, 128), (682, 6, 2, 4, 128), (683, 6, 3, 1, 128), (683, 6, 3, 5, 128),
    # more queries: 4 keys, or queries x keys up to 256 with 512 pairs
    (1, 3, 17, 1, 64), (2, 2, 660, 4, 128), (256, 2, 32, 8, 64), (256, 2, 51, 5, 128),
    (256, 2, 17, 16, 128), (255, 2, 32, 8, 128)])
def test_frame_attention_short_windows(B, H, Lq, Lk, D):
    """The kernel of short windows and the edges of its range, with keys that
    no query, one query or all queries see (a NaN in a row that none sees),
    lanes past the last query and strided q / k / v, against float64.  Bounds
    as in test_frame_attention_edges."""
    need_gpu()
    say("frame attention short windows", B, H, Lq, Lk, D)
    g = torch.Generator("cuda").manual_seed(B + Lq + Lk + D)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16)
    q = rnd(B, Lq + 1, H + 1, D)[:, 1:, 1:]
    k = rnd(B, H, Lk, D).transpose(1, 2)
    v = rnd(B, Lk, 2 * H, D)[:, :, :H]
    kf = (5 + 2 * torch.arange(Lk)) // 3
    qf = 1 + torch.arange(Lq) * (int(kf[-1]) + 2) // Lq
    m = kf[None] <= qf[:, None]
    if Lk > 2:
        m &= qf[:, None] - kf[None] < 4
    dark = ~m.any(0)
    kk, vv = k.clone(), v.clone()
    kk[:, dark], vv[:, dark] = float("nan"), float("inf")
    got = frame_attention(q, kk, vv, qf, kf, 1, 4 if Lk > 2 else -1).double()
    torch.cuda.synchronize()
    t = lambda x: x.double().transpose(1, 2).contiguous()
    sc = t(q) @ t(k).transpose(2, 3).contiguous() / math.sqrt(D)
    p = torch.softmax(sc.masked_fill(~m.cuda(), -math.inf), -1).nan_to_num(0.0)
    ref = (p @ t(v)).transpose(1, 2)
    err = (got - ref).abs()
    assert (err <= 2.0 ** -8 * ref.abs() + 1e-3).all(), float(err.max())
    assert (got[:, (~m.any(1)).cuda()] == 0).all()


class _Attn(nn.Module):
    """The attributes the reference's cached action attention reads."""

    def __init__(self, dim, nh, seed):
        super().__init__()
        torch.manual_seed(seed)
        self.num_heads = nh
        self.q, self.k, self.v, self.o = (nn.Linear(dim, dim) for _ in range(4))
        self.norm_q, self.norm_k = nn.RMSNorm(dim, eps=1e-6), nn.RMSNorm(dim, eps=1e-6)
        for lin in (self.q, self.k, self.v, self.o):
            nn.init.normal_(lin.weight, std=0.05)


def _roped(x, freqs, nh):
    b, s, dim = x.shape
    xc = torch.view_as_complex(x.double().reshape(b, s, nh, -1, 2))
    return torch.view_as_real(xc * freqs).flatten(2).float()


def test_temporal_cached_rollout_matches_full_sequence():
    need_gpu()
    B, T, n, W, nh, hd = 6, 12, 3, 4, 2, 128
    dim = nh * hd
    gpu = _Attn(dim, nh, seed=2).to("cuda", torch.bfloat16)
    ref_attn = copy.deepcopy(gpu).float().cpu()       # the same bf16 weights, in fp32
    g = torch.Generator().manual_seed(3)
    x = torch.randn(B, T, dim, generator=g).to(torch.bfloat16).float()
    freqs = precompute_freqs_cis(hd, end=T).unsqueeze(1)          # [T, 1, hd/2]
    with torch.no_grad():
        qf = _roped(ref_attn.norm_q(ref_attn.q(x)), freqs, nh).view(B, T, nh, hd)
        kf = _roped(ref_attn.norm_k(ref_attn.k(x)), freqs, nh).view(B, T, nh, hd)
        vf = ref_attn.v(x).view(B, T, nh, hd)
    cache = {}
    for b0 in range(0, T, n):
        xb = x[:, b0:b0 + n].to("cuda", torch.bfloat16)
        for rep in range(2):
            say(f"temporal block {b0 // n} pass {rep}")
            with torch.no_grad():
                y = action_temporal_cached_attention(gpu, xb, freqs[b0:b0 + n].cuda(), cache,
                                                     b0, n, W)
            torch.cuda.synchronize()
        m = _temporal(torch.arange(b0, b0 + n), torch.arange(0, b0 + n), n, W)
        att = torch.stack([_sdpa(qf[i, b0:b0 + n], kf[i, :b0 + n], vf[i, :b0 + n], m,
                                 1 / math.sqrt(hd)) for i in range(B)])
        with torch.no_grad():
            ref = ref_attn.o(att.reshape(B, n, dim))
        mx, mn = err_stats(y, ref)
        say(f"  max-abs {mx:.3e} mean-abs {mn:.3e}")
        assert mx <= MAX_ABS and mn <= MEAN_ABS


def test_keyboard_cached_rollout_matches_full_sequence():
    need_gpu()
    B, T, n, W, nh, hd, patches, tpf = 2, 9, 3, 4, 2, 64, 10, 2
    dim = nh * hd
    gpu = _Attn(dim, nh, seed=5).to("cuda", torch.bfloat16)
    ref_attn = copy.deepcopy(gpu).float().cpu()
    g = torch.Generator().manual_seed(6)
    # video tokens and keyboard tokens, frame-major
    xv = torch.randn(B, T * patches, dim, generator=g).to(torch.bfloat16).float()
    kbd = torch.randn(B, T * tpf, dim, generator=g).to(torch.bfloat16).float()
    with torch.no_grad():
        qf = ref_attn.norm_q(ref_attn.q(xv)).view(B, T * patches, nh, hd)
        kf = ref_attn.norm_k(ref_attn.k(kbd)).view(B, T * tpf, nh, hd)
        vf = ref_attn.v(kbd).view(B, T * tpf, nh, hd)
    cache = {}
    for b0 in range(0, T, n):
        xb = xv[:, b0 * patches:(b0 + n) * patches].to("cuda", torch.bfloat16)
        kb = kbd[:, b0 * tpf:(b0 + n) * tpf].to("cuda", torch.bfloat16)
        for rep in range(2):
            say(f"keyboard block {b0 // n} pass {rep}")
            with torch.no_grad():
                y = action_keyboard_cached_attention(gpu, xb, kb, cache, b0, n, W, patches, tpf)
            torch.cuda.synchronize()
        qfr = torch.arange(b0, b0 + n).repeat_interleave(patches)
        kfr = torch.arange(0, (b0 + n) * tpf) // tpf
        m = _temporal(qfr, kfr, n, W)
        att = torch.stack([_sdpa(qf[i, b0 * patches:(b0 + n) * patches], kf[i, :(b0 + n) * tpf],
                                 vf[i, :(b0 + n) * tpf], m, 1 / math.sqrt(hd)) for i in range(B)])
        with torch.no_grad():
            ref = ref_attn.o(att.reshape(B, -1, dim))
        mx, mn = err_stats(y, ref)
        say(f"  max-abs {mx:.3e} mean-abs {mn:.3e}")
        assert mx <= MAX_ABS and mn <= MEAN_ABS
