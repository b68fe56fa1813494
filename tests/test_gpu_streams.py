"""The library keeps no mutable state and enqueues only on the caller's stream:
calls issued from several host threads on several streams at once give the same
results as the same calls made one after the other."""
import threading

import pytest
import torch

import fbcuda_amd as F
from fbcuda_amd import synth
from gpu_util import REGS_NARROW, SMALL, SPLIT, conv_route, dev

pytestmark = pytest.mark.gpu


def work(seed, stream, out, layer):
    B, cin, cout = layer
    d = dev()
    with torch.cuda.stream(stream):
        planes = synth.normal((700, 32, 32), seed=seed, device=d)
        rows = synth.uniform((5000, 128), seed=seed + 1, device=d)
        x = synth.normal((B, cin, 27, 27), seed=seed + 2, device=d)
        w = synth.normal((cout, cin, 5, 5), seed=seed + 3, std=0.05, device=d)
        spec = torch.empty((700, 17, 32, 2), device=d)
        spec1 = torch.empty((5000, 65, 2), device=d)
        y = torch.empty((B, cout, 23, 23), device=d)
        ws = torch.empty(F.conv_workspace(0, B, cin, cout, 32), dtype=torch.uint8, device=d)
        for _ in range(20):
            assert F.fbfft2D(planes, spec, stream=stream) == F.Success
            assert F.fbfft1D(rows, spec1, stream=stream) == F.Success
            assert F.conv_fprop(x, w, y, 32, ws, stream=stream) == F.Success
        stream.synchronize()
        out[seed] = [t.cpu() for t in (spec, spec1, y)]


# a layer without a workspace, and two that hand spectra through theirs
@pytest.mark.parametrize("layer,kind", [((6, 5, 7), SMALL), ((16, 12, 40), REGS_NARROW), ((128, 128, 192), SPLIT)])
def test_concurrent_streams_and_threads(layer, kind):
    assert conv_route(0, 32, *layer, 27, 27, 5)[0] == kind
    seeds = [100, 200, 300, 400]
    serial, parallel = {}, {}
    for s in seeds:
        work(s, torch.cuda.Stream(), serial, layer)
    threads = [threading.Thread(target=work, args=(s, torch.cuda.Stream(), parallel, layer)) for s in seeds]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for s in seeds:
        assert s in parallel
        for a, b in zip(serial[s], parallel[s]):
            assert torch.equal(a, b)
