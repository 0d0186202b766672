"""The state-space convolution of prompts by runs of eight rows, against the plain convolution."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("taps", [2, 3, 4])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads,P,state_size,with_bias", [(4, 16, 20, True), (8, 40, 16, False), (4, 64, 2, True)])
def test_runs_of_rows(taps, dtype, heads, P, state_size, with_bias):
    """Sequences of one row, fewer rows than taps, a run's edges and many rows, some at their
    beginning and some behind an earlier step's tail, a sequence without rows, padding rows in the
    middle and at the end.  Float32 sums of up to four products and a bias: within 2e-6 of the
    float64 result of the same inputs, whose terms are of order one; the tails are copies."""
    from edge_infer_amd.csrc import lib
    torch.manual_seed(taps + heads)
    shape = lib.SsmShape(heads=heads, groups=1, head_dim=P, state=state_size, taps=taps)
    C = shape.channels
    counts, starts = [1, 2, 8, 0, 17, 90, 31], [0, 5, 0, 4, 9, 0, 3]
    row_pos, row_seq, row0s = [], [], []
    for s, (count, start) in enumerate(zip(counts, starts)):
        row0s.append(len(row_pos))
        row_pos += range(start, start + count)
        row_seq += [s] * count
        if s == 4:
            row_pos += [0] * 3
            row_seq += [-1] * 3
    row_pos += [0] * 2
    row_seq += [-1] * 2
    n = len(row_pos)
    assert n >= 128
    proj = torch.randn(n, shape.proj_width).to(dtype)
    w, bias = torch.randn(C, taps) * 0.5, torch.randn(C) * 0.2
    state = torch.randn(2 * len(counts), shape.state_floats)
    tails = state[:, shape.inner * state_size:].reshape(-1, taps - 1, C)
    seq_in, seq_out = list(range(len(counts))), list(range(len(counts), 2 * len(counts)))
    on = state.clone().to(DEV)
    conv = torch.full((n, C), 7.0, device=DEV)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)  # noqa: E731
    lib.ssm_conv(proj.to(DEV), w.to(DEV), bias.to(DEV) if with_bias else None, on, shape, i32(row_pos),
                 i32(row_seq), i32(seq_in), i32(seq_out), i32(starts), i32(counts), i32(row0s), conv)
    conv, on = conv.cpu(), on.cpu()
    assert bool((conv[torch.tensor(row_seq) < 0] == 7.0).all())
    for s, count in enumerate(counts):
        new = on[seq_out[s]][shape.inner * state_size:].reshape(taps - 1, C)
        if count == 0:
            assert torch.equal(on[seq_out[s]], state[seq_out[s]])
            continue
        x = proj[row0s[s]:row0s[s] + count, shape.inner:shape.inner + C].float()
        x = torch.cat([tails[seq_in[s]], x])
        z = sum(w[:, j].double() * x[j:j + count].double() for j in range(taps))
        z = z + (bias.double() if with_bias else 0.0)
        want = z * torch.sigmoid(z)
        assert (conv[row0s[s]:row0s[s] + count].double() - want).abs().max().item() <= 2e-6 * max(
            1.0, want.abs().max().item())
        assert torch.equal(new, x[-(taps - 1):])
