"""GPU tests of what a decode step does once in front of its layers: the launch that stages a graph's inputs, and the shared-prefix plan of a
batch that is compared and planned by one workgroup (up to 16 requests) or by two launches (above)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("given,padded", [(1, 1), (1, 2), (63, 64), (64, 64), (255, 256), (257, 288), (0, 8)])
@pytest.mark.parametrize("own", [(), (1, 3), (0, 1, 2, 3)])
def test_stage_decode_inputs(device, given, padded, own):
    from sglang_amd import kernels as K

    types = (torch.int64, torch.int64, torch.int32, torch.int64)
    bufs = [torch.randint(1, 1000, (padded + 3,), device=device).to(t) for t in types]
    src = [b[:given] if i in own else torch.randint(1, 1000, (given,), device=device).to(t) for i, (b, t) in enumerate(zip(bufs, types))]
    want = [torch.cat([s, torch.full((padded - given,), 5 if i == 2 else 0, dtype=t, device=device), b[padded:]])
            for i, (s, b, t) in enumerate(zip(src, bufs, types))]
    assert K.stage_decode_inputs(src, bufs, given, padded, 5)
    for w, b in zip(want, bufs):
        assert torch.equal(w, b)


def test_stage_decode_inputs_leaves_the_rest_to_copies(device):
    from sglang_amd import kernels as K

    bufs = [torch.zeros(8, dtype=t, device=device) for t in (torch.int64, torch.int64, torch.int32, torch.int64)]
    good = [torch.ones(4, dtype=b.dtype, device=device) for b in bufs]
    for i, bad in ((2, good[2].long()), (0, torch.ones(8, dtype=torch.int64, device=device)[::2]), (1, good[1][:3]), (3, good[3].cpu())):
        src = list(good)
        src[i] = bad
        assert not K.stage_decode_inputs(src, bufs, 4, 8, 1)
    assert all(int(b.abs().sum()) == 0 for b in bufs)


@pytest.mark.parametrize("n", [2, 3, 15, 16])
@pytest.mark.parametrize("shared", [127, 128, 640, 2500])
def test_plan_of_one_launch_equals_two(device, n, shared):
    """The same requests, and with 17 - n requests of one token behind them: the plan's two launches."""
    from sglang_amd import kernels as K

    g = torch.Generator().manual_seed(n + shared)
    B, width = 17, 4096
    lens = [shared + int(torch.randint(1, 300, (1,), generator=g)) for _ in range(n)] + [1] * (B - n)
    r2t = torch.arange(1, 1 + (B + 1) * width, dtype=torch.int32).view(B + 1, width)
    for b in range(n):
        r2t[b + 1, :shared] = r2t[1 + b % 2, :shared]                # two groups
    if n > 2:
        r2t[3, shared // 2] = 999999                                 # one member leaves its group early
    r2t, pool = r2t.to(device), torch.arange(1, B + 1, device=device)
    seen = []
    for count in (n, B):
        seq = torch.tensor(lens[:count], dtype=torch.int32, device=device)
        ws = K.CascadeWorkspace(count, 32, 128, width, device)
        K.cascade_plan(ws, r2t, pool[:count], seq, 32, 8)
        s = K.cascade_plan_summary(ws, count)
        rows = [i for i in s["private_items"] if i[0] < n]
        seen.append((s["n_shared_items"], s["n_groups"], s["req_shared"][:n], s["member_rows"], s["group_qo"], s["group_pool_row"], s["group_kvlen"],
                     s["items"], rows, [b for b in s["batch_order"] if b < n]))
    assert seen[0] == seen[1]
