"""Graph captures for test_captured_backward_repeats, test_graphed_modules_train and
test_masked_block_under_capture_is_an_error, in a process of their own: a program captures on its own streams, and
what a capture leaves behind stays out of the other tests.  Prints a line for each case, ends with status 1 after a mismatch."""

import sys

import torch

from oracle import rglru_oracle as orc
from tests.helpers import PARAMS, rel_err


def _layer(dtype, shape):
    from griffin_amd import hip_rglru

    case = orc.make_case(*shape, seed=11)
    leaves = [case[k].to(dtype).cuda().requires_grad_(True) for k in PARAMS]
    return leaves, lambda: hip_rglru(*leaves, 8.0)[0]


def _scan(dtype, shape):
    from griffin_amd import hip_rglru_scan

    B, T, W = shape
    g = torch.Generator().manual_seed(2)
    a = torch.sigmoid(torch.randn(B, T, W, generator=g) + 2.0)
    leaves = [t.cuda().requires_grad_(True) for t in (a, torch.randn(B, T, W, generator=g), torch.randn(B, W, generator=g))]
    return leaves, lambda: hip_rglru_scan(*leaves)


def _block(dtype, shape):
    from griffin_amd import RecurrentBlock

    B, T, D, W, nb = shape
    torch.manual_seed(5)
    block = RecurrentBlock(D, W, gate_blocks=nb, scan_mode="hip").to(dtype).cuda()
    x = torch.randn(B, T, D).to(dtype).cuda().requires_grad_(True)
    return [x, *block.parameters()], lambda: block(x)


# each path that clears records: portable kernels, tiles with look-back, wide blocks, the bare scan, the block as one node
CASES = [
    ("portable", _layer, torch.float32, (2, 70, 48, 3), 1e-5),
    ("tiled", _layer, torch.bfloat16, (2, 200, 256, 2), 2e-2),
    ("wide", _layer, torch.bfloat16, (2, 200, 320, 2), 2e-2),
    ("scan", _scan, torch.float32, (2, 300, 130), 1e-5),
    ("scan, four channels to a lane", _scan, torch.float32, (2, 300, 256), 1e-5),
    ("block", _block, torch.bfloat16, (2, 200, 64, 256, 2), 2e-2),
]


def captured_backward(make, dtype, shape, tol):
    """A graph of the backward pass alone, the first one over an eager forward, replayed for several upstream gradients."""
    leaves, forward = make(dtype, shape)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        y = forward()
        ups = [torch.randn(y.shape, generator=torch.Generator().manual_seed(i)).to(dtype).cuda() for i in range(3)]
        want = [[g.clone() for g in torch.autograd.grad(y, leaves, up, retain_graph=True)] for up in ups]
        dy = ups[0].clone()
        y = forward()                                        # nothing has gone back over this one yet
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        got = torch.autograd.grad(y, leaves, dy, retain_graph=True)
    worst = 0.0
    for up, expected in zip(ups, want):
        dy.copy_(up)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        worst = max([worst] + [rel_err(a.float(), b.float()) for a, b in zip(got, expected)])
    # the same graph of the autograd engine again, eagerly
    again = torch.autograd.grad(y, leaves, ups[0])
    torch.cuda.synchronize()
    worst = max([worst] + [rel_err(a.float(), b.float()) for a, b in zip(again, want[0])])
    return worst, worst < tol


def graphed_modules():
    """torch.cuda.make_graphed_callables: forward and backward in graphs of their own, replayed as a training loop does."""
    from griffin_amd import RG_LRU, RecurrentBlock

    ok = True
    for name, make, shape, dtype, tol in (("layer", lambda: RG_LRU(96, gate_blocks=3), (2, 70, 96), torch.float32, 1e-5),
                                          ("layer", lambda: RG_LRU(256, gate_blocks=2), (2, 200, 256), torch.bfloat16, 2e-2),
                                          ("block", lambda: RecurrentBlock(64, 256, gate_blocks=2), (2, 200, 64), torch.bfloat16, 2e-2)):
        print("graphed module", name, shape, flush=True)
        torch.manual_seed(7)
        plain = make().to(dtype).cuda()
        graphed = make().to(dtype).cuda()
        graphed.load_state_dict(plain.state_dict())
        graphed = torch.cuda.make_graphed_callables(graphed, (torch.randn(*shape, device="cuda", dtype=dtype, requires_grad=True),))
        worst = 0.0
        for _ in range(3):
            x, dy = (torch.randn(*shape, device="cuda", dtype=dtype) for _ in range(2))
            results = []
            for module in (plain, graphed):
                module.zero_grad(set_to_none=True)
                leaf = x.clone().requires_grad_(True)
                y = module(leaf)
                y.backward(dy)
                torch.cuda.synchronize()
                results.append([y.detach().clone(), leaf.grad.clone(), *(p.grad.clone() for p in module.parameters())])
            worst = max([worst] + [rel_err(b.float(), a.float()) for a, b in zip(*results)])
        print("  worst", "%.2e" % worst, flush=True)
        ok &= worst < tol
    return ok


def captured_mask():
    """Which kernels a masked block runs is decided on the host: under capture that is a RuntimeError before anything is
    launched, the process goes on, and the same call outside the capture is what it was."""
    from griffin_amd import RecurrentBlock

    ok = True
    for dtype in (torch.bfloat16, torch.float32):
        torch.manual_seed(5)
        block = RecurrentBlock(64, 128, gate_blocks=2, scan_mode="hip").to(dtype).cuda()
        x = torch.randn(2, 40, 64).to(dtype).cuda()
        mask = torch.ones(2, 40, dtype=torch.bool, device="cuda")
        mask[1, 17:] = False
        for train in (False, True):
            with torch.set_grad_enabled(train):
                want = block(x, active_mask=mask).detach()
                torch.cuda.synchronize()
                try:
                    with torch.cuda.graph(torch.cuda.CUDAGraph()):
                        block(x, active_mask=mask)
                    ok = False
                except RuntimeError as error:
                    print("  refused:", str(error).splitlines()[0], flush=True)
                torch.cuda.synchronize()
                ok &= rel_err(block(x, active_mask=mask).float(), want.float()) < 1e-2
    return ok


def captured_backwards():
    ok = True
    for name, make, dtype, shape, tol in CASES:
        print("captured backward", name, shape, flush=True)
        worst, good = captured_backward(make, dtype, shape, tol)
        print("  worst", "%.2e" % worst, flush=True)
        ok &= good
    return ok


if __name__ == "__main__":
    sys.exit(0 if {"backward": captured_backwards, "modules": graphed_modules, "mask": captured_mask}[sys.argv[1]]() else 1)
