"""The K-split decode-GEMM (exl3_gemm and exl3_gemm_grouped at 17..512 rows): the CPU address
replay over its tile, ring and split edges, and GPU parity with the fp64 oracle at the same edges.

Bar: per-row relative L2 error <= 1e-3 against the oracle on the same fp16 inputs (activations and
weights each rounded to 11 bits, sums in fp32: 3e-4 expected).
"""
import ctypes
import os
import random

import pytest
import torch

from orcasaq2 import synthetic as syn

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "orcasaq2-kernel_amd", "orcasaq2", "libexl3replay.so")
REL_TOL = 1e-3


@pytest.fixture(scope="module")
def replay():
    lib = ctypes.CDLL(LIB)
    lib.exl3r_message.restype = ctypes.c_char_p

    def run(rows, ic, ocs, Ks, cbs, cus):
        arr = lambda v: (ctypes.c_int * len(v))(*v)  # noqa: E731
        st = (ctypes.c_longlong * 4)()
        rc = lib.exl3r_gemm_ks(rows, ic, len(ocs), arr(ocs), arr(Ks), arr(cbs), cus, st)
        assert rc == 0, (rows, ic, ocs, Ks, cbs, cus, lib.exl3r_message().decode())
        return list(st)
    return run


# row tiles of 32..128 rows, one to four of them; below 17 rows the entry point takes any count
@pytest.mark.parametrize("rows", [1, 17, 32, 33, 64, 65, 96, 97, 128, 129, 200, 256, 257, 384, 512])
def test_replay_layers(replay, rows):
    for cus in (256, 80, 3):
        assert replay(rows, 5120, [6144, 1024, 1024], [4, 5, 3], [0, 0, 0], cus)[0] == 1
    replay(rows, 2048, [2048], [4], [1], 256)
    replay(rows, 128, [128], [1], [0], 256)


def test_replay_random_shapes(replay):
    rnd = random.Random(8101)
    for _ in range(80):
        n = rnd.randint(1, 9)
        replay(rnd.randint(1, 512), 128 * rnd.randint(1, 24), [128 * rnd.randint(1, 20) for _ in range(n)],
               [rnd.randint(1, 8) for _ in range(n)], [rnd.randint(0, 1) for _ in range(n)],
               rnd.choice((256, 304, 80, 8, 1, 2, 33)))


# ic = 128 (four steps) leaves pairs without steps; 1152 and 3200 inputs leave uneven runs; more
# column groups than workgroups (oc = 33024: 258) give a whole round and a split one
@pytest.mark.gpu
@pytest.mark.parametrize("rows,ic,spec", [
    (17, 128, [(128, 1, 0)]),
    (32, 1152, [(384, 2, 1), (128, 7, 1)]),
    (33, 3200, [(256, 3, 0), (128, 6, 0), (128, 8, 0)]),
    (64, 1152, [(1280, 5, 0)]),
    (97, 640, [(33024, 2, 0)]),
    (128, 3200, [(256, 4, 1), (256, 5, 1)]),
    (129, 1152, [(384, 3, 0)]),
    (257, 640, [(512, 1, 1), (128, 6, 1)]),
    (512, 1152, [(256, 7, 0), (128, 8, 0)]),
])
def test_gpu_edges(native, oracle, rows, ic, spec):
    print(f"K-split GEMM rows={rows} ic={ic} {spec}", flush=True)
    dev = torch.device("cuda", 0)
    lins = [syn.linear(ic, oc, K, seed=31 * rows + i) for i, (oc, K, _) in enumerate(spec)]
    x = syn.activations(rows, ic, torch.Generator().manual_seed(rows))
    shards = [dict(trellis=l["trellis"].to(dev), suh=l["suh"].to(dev), svh=l["svh"].to(dev), oc=oc, K=K, codebook=cb)
              for l, (oc, K, cb) in zip(lins, spec)]
    y = native.gemm_grouped(x.to(dev), shards)
    assert torch.equal(native.gemm_grouped(x.to(dev), shards), y)
    # sampled rows (every tile's first and last) of all columns
    pick = sorted({r for r in (0, 31, 32, 63, 64, 127, 128, 255, 256, rows // 2, rows - 1) if r < rows})
    col = 0
    for l, (oc, K, cb) in zip(lins, spec):
        ref = oracle.shard_gemm_ref(x[pick].numpy(), l["trellis"], l["suh"].numpy(), l["svh"].numpy(), K, cb)
        err = oracle.rel_err_rows(y[pick, col:col + oc].float().cpu().numpy(), ref)
        assert err.max() <= REL_TOL, (oc, K, cb, err.max())
        col += oc
