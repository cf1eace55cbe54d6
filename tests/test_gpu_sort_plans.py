"""The radix sort's plans (threads and keys per thread, digit width by the number of keys) at their edges."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from gswarp_amd import _lib
from test_gpu_sort import _field, _keys, _sort


@pytest.mark.gpu
@pytest.mark.parametrize("n", [2047, 2048, 2049, 4097, 786_432, 786_433, 2_097_152, 2_097_153])
@pytest.mark.parametrize("name,key_bits", [("gs_sort_keys_u64", 13), ("gs_sort_pairs_u32", 26)])
def test_plan_edges(name, key_bits, n, device):
    rng = np.random.default_rng(n)
    keys = _keys(n, "uniform", rng, np.uint64 if name.endswith("u64") else np.uint32)
    vals = rng.permutation(n).astype(np.int32) if "pairs" in name else None
    out_k, out_v = _sort(name, n, 0, key_bits, keys, vals, device)
    order = np.argsort(_field(keys, 0, key_bits), kind="stable")
    assert np.array_equal(out_k, keys[order])
    assert vals is None or np.array_equal(out_v, vals[order])


@pytest.mark.gpu
@pytest.mark.parametrize("n", [5000, 1_000_000])
def test_scratch_for_4096_key_tiles_is_enough(n, device):
    """One column of 256 counters per 4096 keys and the digit totals, as little as any size needs."""
    lib = _lib.load()
    need = ((((n + 4095) // 4096 + 1) * 1024) + 255) & ~255
    assert need < lib.gs_sort_scratch_bytes(n)
    keys = _keys(n, "uniform", np.random.default_rng(n), np.uint64)
    kt = torch.from_numpy(keys.view(np.int64)).to(device)
    alt = torch.empty_like(kt)
    scratch = torch.empty((need,), dtype=torch.uint8, device=device)
    stream = torch.cuda.current_stream(device).cuda_stream
    lib.call("gs_sort_keys_u64", n, 0, 16, kt.data_ptr(), alt.data_ptr(), scratch.data_ptr(), need, stream)
    torch.cuda.synchronize()
    assert np.array_equal(kt.cpu().numpy().view(np.uint64), keys[np.argsort(_field(keys, 0, 16), kind="stable")])
    raw = lib.gs_sort_keys_u64
    assert raw(n, 0, 16, kt.data_ptr(), alt.data_ptr(), scratch.data_ptr(), need - 256, stream) != 0


def test_scratch_never_falls():
    lib = _lib.load()
    sizes = [1, 2048, 4096, 786_432, 786_433, 1_572_864, 1_572_865, 2_097_152, 2_097_153, 9_000_000, 1 << 24, 1 << 28]
    got = [lib.gs_sort_scratch_bytes(n) for n in sizes]
    assert got == sorted(got)
