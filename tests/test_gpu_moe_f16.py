"""GPU parity of the unquantized grouped GEMM drop-in (moe_grouped_gemm).

The reference kernel rounds both operands to fp16, sums in fp32 and stores fp16
(src/kernels.py:440-523).  The oracle sums the fp16-rounded operands exactly (fp64), so
the device result may differ from it by the fp32 summation error plus the fp16 store:
normwise max relative error <= 1e-3 (the fp16 step is 2^-11 relative).
"""
import pytest
import torch
import torch.nn.functional as F

from oracle import fp8_oracle as orc

pytestmark = pytest.mark.gpu


def test_reference_equivalence(kern, dev):
    """The reference's own test (tests/test_kernels.py:131-155), same shapes and bound."""
    n_experts, d_model, hidden_dim, total_tokens = 8, 512, 128, 256
    g = torch.Generator().manual_seed(0)
    weights = torch.randn(n_experts, hidden_dim, d_model, generator=g).to(torch.bfloat16)
    sorted_x = torch.randn(total_tokens, d_model, generator=g).to(torch.bfloat16)
    per = total_tokens // n_experts
    starts = torch.arange(0, total_tokens, per)[:n_experts]
    ends = torch.cat([starts[1:], torch.tensor([total_tokens])])
    out = kern.moe_grouped_gemm(sorted_x.to(dev), weights.to(dev), starts.to(dev), ends.to(dev))
    assert out.shape == (total_tokens, hidden_dim) and out.dtype == torch.float16
    ref = torch.zeros(total_tokens, hidden_dim)
    for i in range(n_experts):
        s, t = int(starts[i]), int(ends[i])
        ref[s:t] = F.linear(sorted_x[s:t].float(), weights[i].float())
    rel = (ref - out.float().cpu()).abs() / (ref.abs() + 1e-6)
    assert rel.mean().item() < 0.01


@pytest.mark.parametrize("xdt,wdt", [(torch.bfloat16, torch.float32), (torch.float16, torch.float16),
                                     (torch.float32, torch.bfloat16)])
@pytest.mark.parametrize("N,K", [(384, 512), (100, 200)])
def test_grouped_f16_parity(kern, dev, xdt, wdt, N, K):
    counts = [300, 0, 128, 1, 555, 64, 0, 1000]
    ends = torch.tensor(counts).cumsum(0)
    starts = ends - torch.tensor(counts)
    T, E = int(ends[-1]), len(counts)
    g = torch.Generator().manual_seed(N + K)
    x = torch.randn(T, K, generator=g).to(xdt)
    w = (torch.randn(E, N, K, generator=g) * 0.05).to(wdt)
    out = kern.moe_grouped_gemm(x.to(dev), w.to(dev), starts.to(dev), ends.to(dev)).float().cpu()
    ref = orc.grouped_gemm_f16_ref(x, w, starts, ends)
    inside = torch.zeros(T, dtype=torch.bool)
    for _, s, t in orc.expert_slices(starts, ends, T):
        inside[s:t] = True
    got, want = out[inside].double(), ref[inside]
    assert (got - want).abs().max() / want.abs().max() <= 1e-3


# Every tile (64 x 128, 128 x 128, 256 x 256): partial rows, columns and K steps, one K step,
# experts without rows, more than 64 experts, odd K; and against rows that start anywhere
# (loaded without alignment), whose sums are the same in the same order
@pytest.mark.parametrize("counts,N,K", [
    ([3, 0, 65, 1, 40], 136, 8), ([2] * 66 + [0, 100], 200, 200),
    ([300, 0, 128, 1, 555, 64, 0, 1000], 328, 520),
    ([9000, 0, 257, 7127, 1], 2120, 72),
    ([300, 0, 70, 5], 100, 131), ([2] * 66 + [100], 64, 7), ([700, 300], 130, 1),
])
@pytest.mark.parametrize("xdt,wdt", [(torch.bfloat16, torch.float32), (torch.float16, torch.bfloat16),
                                     (torch.float32, torch.float16)])
def test_grouped_f16_tiles(kern, dev, counts, N, K, xdt, wdt):
    ends = torch.tensor(counts).cumsum(0).to(dev)
    starts = ends - torch.tensor(counts, device=dev)
    T, E = sum(counts), len(counts)
    g = torch.Generator(device=dev).manual_seed(N + K)
    x = torch.randn(T, K, generator=g, device=dev).to(xdt)
    w = (torch.randn(E, N, K, generator=g, device=dev) * 0.05).to(wdt)
    out = kern.moe_grouped_gemm(x, w, starts, ends)
    wide = torch.zeros(T, K + 1, dtype=xdt, device=dev)
    wide[:, :K] = x
    general = kern.moe_grouped_gemm(wide[:, :K], w, starts, ends)
    assert torch.equal(out, general)
    # fp32 sums of exact fp16 products (2^-24 a term) and one fp16 rounding (2^-11)
    want = torch.cat([x[a:b].half().double() @ w[e].half().double().t()
                      for e, (a, b) in enumerate(zip(starts.tolist(), ends.tolist()))])
    assert ((out.double() - want).abs() <= 2 ** -10 * want.abs() + K * 2 ** -22 * want.abs().max()).all()
