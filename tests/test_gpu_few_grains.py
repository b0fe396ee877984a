"""ri_LROT at the sizes where its kernels change: waves of 64 grains and their
remainders, even and odd row lengths, the 32-step chunks of the kinematics, the
line between few and many grains; against the defining Euler step in float64."""
import pytest

pytestmark = pytest.mark.gpu


def plain(ri0, dt, Nt, D, W, iota):
    import torch
    r, out = ri0, [ri0]
    for t in range(Nt - 1):
        Dr = r @ D[t].T
        r = r + dt * (r @ W[t].T + iota * (r * (r * Dr).sum(1, keepdim=True) - Dr * (r * r).sum(1, keepdim=True)))
        r = r / r.norm(dim=1, keepdim=True)
        out.append(r)
    return torch.stack(out)


@pytest.mark.parametrize("N,Nt", [(1, 1), (1, 2), (2, 33), (63, 32), (64, 34), (65, 65), (130, 97), (64 * 1280 - 1, 3),
                                  (64 * 1280, 4), (64 * 1280 + 1, 3), (64 * 1280 + 2, 2)])
def test_few_grains_edges(gpu_ctx, N, Nt):
    import torch
    from specfab_amd import batch as B
    g = torch.Generator(device="cuda").manual_seed(N + Nt)
    r0 = torch.randn((N, 3), generator=g, device="cuda", dtype=torch.float64)
    r0 = 1.3 * r0 / r0.norm(dim=1, keepdim=True)     # not of unit length: rounded off by the first step
    D, W = (torch.randn((Nt, 3, 3), generator=g, device="cuda", dtype=torch.float64) for _ in range(2))
    out = B.ri_LROT_batch(r0, 0.02, Nt, D, W, 0.9)
    ref = plain(r0, 0.02, Nt, D, W, 0.9)
    # a few rounding errors of 1.1e-16 per step, carried over at most 97 steps
    assert out.shape == ref.shape and (out - ref).abs().max().item() < 1e-13
