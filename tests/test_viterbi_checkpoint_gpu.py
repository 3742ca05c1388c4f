"""The checkpointed traceback of the tile Viterbi (K2..K4): contexts that end
its segments at every depth, and equality with the recorded decisions (which
a workspace too small for the checkpoints selects) on costs that tie,
saturate, overflow or are not numbers."""

from __future__ import annotations

import sys

import numpy as np
import pytest
import torch

from conftest import device_memory_left
from oracle import tables as otables
from oracle import viterbi as ov
from qsrt_amd import _native
from qsrt_amd.sqg_e4m3 import sqg_xor_cheb_t12_bytes
from qsrt_amd.sqg_quantizer import viterbi_tiles

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("context", (2, 3, 4, 5, 6, 7, 126, 127))
@pytest.mark.parametrize("bits", (2, 3, 4))
def test_every_bottom_segment_matches_oracle(bits, context):
    lag = context & 1
    print(f"[viterbi] K{bits} C{context} lag{lag}: 20 tiles", file=sys.stderr, flush=True)
    tiles = np.random.default_rng(1000 * bits + context).standard_normal((20, 256)).astype(np.float32)
    tiles[4] = 0.0
    tiles[9] *= 100.0
    recon, states = viterbi_tiles(torch.from_numpy(tiles).cuda(), sqg_xor_cheb_t12_bytes(bits).cuda(), bits,
                                  tailbite_context=context, lag=lag)
    o_recon, o_states = ov.encode(tiles, otables.t12_values(bits), K=bits, context=context, boundary_lag=lag)
    assert np.array_equal(states.cpu().numpy().view(np.uint16), o_states)
    assert np.array_equal(recon.cpu().numpy(), o_recon)


@pytest.mark.parametrize("bits", (2, 3, 4))
def test_checkpoints_equal_recorded_decisions(bits):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    n = cus + 44  # more tiles than workgroups: both kernels walk several
    print(f"[viterbi] K{bits}: {n} tiles through both tracebacks", file=sys.stderr, flush=True)
    rng = np.random.default_rng(70 + bits)
    tiles = (rng.standard_normal((n, 256)) * 1.2).astype(np.float32)
    labels = otables.t12_values(bits).astype(np.float32)
    tiles[10:20] = rng.choice(labels[rng.integers(0, 65536, 3)], size=(10, 256))  # exact ties
    tiles[20] = 1e8    # every edge of a step costs the same
    tiles[21] = 1e4
    tiles[22, 100] = 1e30  # overflows: infinite from there on
    tiles[23, 255] = np.inf
    tiles[24, 3] = -np.inf
    tiles[25, 128] = np.nan
    tiles[26] = 1.3e18  # the sum overflows part of the way
    tiles[27] *= 1e-30
    gpu, lut = torch.from_numpy(tiles).cuda(), sqg_xor_cheb_t12_bytes(bits).cuda()
    lag = 0 if bits == 2 else 1
    recon, states = viterbi_tiles(gpu, lut, bits, lag=lag)
    lib = _native.lib()
    small = cus * (1 << 20 if bits == 4 else 1 << 21)  # two decision buffers for each workgroup
    assert small < lib.qsrt_viterbi_workspace_bytes(bits, n)
    workspace = torch.empty(small, dtype=torch.uint8, device="cuda")
    r2, s2 = torch.empty_like(recon), torch.empty_like(states)
    _native.check(lib.qsrt_viterbi_tiles(gpu.data_ptr(), r2.data_ptr(), s2.data_ptr(), n, bits, 128, lut.data_ptr(), lag,
                                         workspace.data_ptr(), small, _native.stream_handle(gpu.device)),
                  "qsrt_viterbi_tiles")
    differ = (states != s2).any(dim=1).nonzero().flatten().tolist()
    assert not differ, f"tiles {differ[:8]} differ"
    assert torch.equal(recon, r2)


@pytest.mark.parametrize("bits,n,cap", [(4, 1, 0), (2, 3, 0), (3, 300, 10), (4, 300, 0)])
def test_workspace_is_sized_by_the_launch_and_given_back(bits, n, cap):
    """A call takes what its own rate and grid use, and holds none of it afterwards."""

    print(f"[viterbi] K{bits}: {n} tiles on at most {cap} workgroups, memory", file=sys.stderr, flush=True)
    tiles = torch.randn((n, 256), device="cuda")
    lut = sqg_xor_cheb_t12_bytes(bits).cuda()
    with torch.cuda.stream(torch.cuda.Stream()):
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        out = viterbi_tiles(tiles, lut, bits, max_workgroups=cap)
        torch.cuda.synchronize()
        peak = torch.cuda.max_memory_allocated() - before
        kept = torch.cuda.memory_allocated() - before
    results = 2 * 512 + sum(t.numel() * t.element_size() for t in out)  # blocks of the allocator are whole 512 bytes
    assert kept <= results
    # and a large one is not cut where 1 MiB or less would be left over
    assert peak <= results + (1 << 20) + _native.lib().qsrt_viterbi_workspace_bytes(bits, cap or n)


@pytest.mark.parametrize("bits", (2, 3, 4))
def test_checkpoints_that_do_not_fit_give_way_to_recorded_decisions(bits):
    n = 300
    print(f"[viterbi] K{bits}: {n} tiles, memory for the recorded decisions only", file=sys.stderr, flush=True)
    tiles = torch.randn((n, 256), device="cuda")
    lut = sqg_xor_cheb_t12_bytes(bits).cuda()
    recon, states = viterbi_tiles(tiles, lut, bits)
    recorded = torch.cuda.get_device_properties(0).multi_processor_count * (1 << 20 if bits == 4 else 2 << 20)
    assert recorded < _native.lib().qsrt_viterbi_workspace_bytes(bits, n)
    with device_memory_left(recorded + (64 << 20)), torch.cuda.stream(torch.cuda.Stream()):  # 64 MiB for the results
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        r2, s2 = viterbi_tiles(tiles, lut, bits)
        assert torch.cuda.max_memory_allocated() - before < recorded + (64 << 20)
    assert torch.equal(states, s2) and torch.equal(recon, r2)


@pytest.mark.parametrize("bits", (2, 4))
def test_captured_launch_keeps_its_workspace(bits):
    """Replays with launches of the program's own in between, wider and narrower ones: each equals the eager result."""

    n = 40
    print(f"[viterbi] K{bits}: {n} tiles in a graph", file=sys.stderr, flush=True)
    tiles = torch.randn((n, 256), device="cuda")
    lut = sqg_xor_cheb_t12_bytes(bits).cuda()
    want, want_states = viterbi_tiles(tiles, lut, bits)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        recon, states = viterbi_tiles(tiles, lut, bits)
    for other in (300, 1, 600):
        recon.zero_()
        states.zero_()
        side = torch.randn((other, 256), device="cuda")
        first = viterbi_tiles(side, lut, bits)
        graph.replay()
        again = viterbi_tiles(side, lut, bits)
        torch.cuda.synchronize()
        assert torch.equal(states, want_states) and torch.equal(recon, want)
        assert torch.equal(first[1], again[1])
