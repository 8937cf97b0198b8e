"""The attention forward kernel in every division of its work (one or two parts of the keys, 64 or 128 queries
to a workgroup), with as few and as many key tiles as each takes: fewer tiles than parts, an odd one over, a
last tile and a last workgroup that are nearly empty."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [(1, 1, 1), (1, 2, 63), (2, 3, 64), (1, 4, 65), (1, 4, 129), (2, 8, 192), (1, 8, 449),      # 64 queries, two parts
         (4, 16, 321), (4, 16, 449), (3, 16, 512), (6, 16, 577),                                    # 128 queries, two parts
         (18, 16, 193), (16, 16, 320), (40, 16, 65), (9, 16, 513)]                                  # 128 queries, one part


@pytest.mark.parametrize("causal", [0, 1])
@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("B,H,S", CASES)
def test_forward(hip, B, H, S, hd, causal):
    from nabla_amd.backend import lib
    gen = torch.Generator(device="cuda").manual_seed(S + hd)
    q, k, v = ((torch.randn(B, S, H, hd, generator=gen, device="cuda") * s).bfloat16() for s in (1.5, 1.5, 1.0))
    k[:, S // 2] *= 4  # (a maximum that one part alone sees)
    guard = 3.0
    o = torch.full((B, S + 1, H, hd), guard, device="cuda", dtype=torch.bfloat16)
    lo, lse = torch.full_like(o, guard), torch.full((B * H * S + 1,), guard, device="cuda")
    d = lib.AttnDesc()
    d.B, d.H, d.S, d.hd, d.scale, d.causal, d.dtype, d.any_length = B, H, S, hd, hd ** -0.5, causal, 1, 1

    def tensor(t):
        a = lib.AttnTensor()
        a.ptr, a.sb, a.ss, a.sh = t.data_ptr(), t.stride(0), t.stride(1), t.stride(2)
        return a

    ts = [tensor(t) for t in (q, k, v, o, lo)]
    lib.check(lib.load().nbk_attention_fwd(C.byref(d), *[C.byref(t) for t in ts], C.c_void_p(lse.data_ptr()),
                                           C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    qf, kf, vf = (t.float().transpose(1, 2).contiguous() for t in (q, k, v))
    s = torch.matmul(qf, kf.transpose(2, 3).contiguous()) * hd ** -0.5
    if causal:
        s = s.masked_fill(torch.ones(S, S, device="cuda", dtype=torch.bool).triu(1), float("-inf"))
    want = torch.matmul(torch.softmax(s, -1), vf).transpose(1, 2)
    got = o[:, :S].float() + lo[:, :S].float()
    # probabilities are rounded to bf16 (2^-9 of each) and normalised by their rounded sum; the result keeps 16 bits
    assert (got - want).norm() <= 2.0 ** -8 * want.norm()
    assert ((got - want).abs() <= 2.0 ** -7 * vf.abs().amax()).all()
    assert (lse[:-1].view(B, H, S) - torch.logsumexp(s, -1)).abs().max() <= 2e-5
    assert lse[-1] == guard and (o[:, S] == guard).all() and (lo[:, S] == guard).all()
