"""The per-element tables of a tiled layout made on the device
(layout_kernels.hip): the row-start flags and a split layout's position map,
entry for entry what their definition (tile_layout.h) gives.  The host's
tables of the same definition are decoded under the sanitizers by
test_tile_layout.py."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

P, U64 = C.c_void_p, C.c_uint64


def _launcher(name, *types):
    from cdmf_amd import solver
    f = getattr(solver.hip_lib(), name)
    f.restype, f.argtypes = C.c_int, types
    return f


def _device(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int32)).cuda()


def _lengths(kind, seed):
    r = np.random.default_rng(seed)
    return {"one": [1], "whole_tiles": [512, 512, 1024, 2048], "long": [5000, 1, 0, 3, 20000],
            "holes": np.where(r.random(900) < 0.4, 0, r.integers(1, 40, 900)),
            "empty": [0, 0, 0], "short": r.integers(0, 4, 40000), "many": r.integers(1, 3, 1 << 20)}[kind]


KINDS = ["one", "whole_tiles", "long", "holes", "empty", "short", "many"]


def _ptr(lengths):
    return np.concatenate([[0], np.cumsum(lengths)]).astype(np.uint32)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("sigma", [8, 16, 24, 32])
def test_row_start_flags(kind, sigma):
    """One word a lane, 16 bits up to sigma 16: bit e % sigma of lane
    e / sigma for every row's first element e."""
    import torch
    launch = _launcher("_ZN3ccd17launch_tile_flagsEPKjmmiPjP12ihipStream_t", P, U64, U64, C.c_int, P, P)
    lengths = np.asarray(_lengths(kind, sigma))
    ptr = _ptr(lengths)
    ntiles = -(-int(ptr[-1]) // (64 * sigma))
    want = np.zeros(64 * ntiles, np.uint32)
    start = ptr[:-1][lengths > 0].astype(np.int64)
    np.bitwise_or.at(want, start // sigma, np.uint32(1) << (start % sigma).astype(np.uint32))
    want = want.astype(np.uint16) if sigma <= 16 else want
    dptr, out = _device(ptr), torch.full((64 * max(ntiles, 1) + 1,), -1, dtype=torch.int32, device="cuda")
    assert launch(dptr.data_ptr(), lengths.size, ntiles, sigma, out.data_ptr(), None) == 0
    torch.cuda.synchronize()
    got = out.cpu().numpy().view(want.dtype)
    assert np.array_equal(got[:want.size], want)
    assert np.all(got[want.size:] == np.iinfo(want.dtype).max)  # nothing past the tiles


@pytest.mark.parametrize("kind", KINDS)
def test_split_positions(kind):
    """All rows' first parts (below[r] elements), then the rest of each row
    that has one, in row order."""
    import torch
    launch = _launcher("_ZN3ccd22launch_split_positionsEPKjmS1_S1_S1_jPjP12ihipStream_t", P, U64, P, P, P, C.c_uint32, P,
                       P)
    lengths = np.asarray(_lengths(kind, 3)).astype(np.int64)
    r = np.random.default_rng(4)
    below = np.minimum(lengths, r.integers(0, np.maximum(lengths, 1) * 2 + 1))  # none, some and all of a row
    ptr, m = _ptr(lengths), lengths.size
    cold = np.flatnonzero(below < lengths).astype(np.uint32)
    vptr = _ptr(np.concatenate([below, (lengths - below)[cold]]))
    src = np.concatenate([ptr[:-1].astype(np.int64), ptr[cold].astype(np.int64) + below[cold]])
    want = np.repeat(src - vptr[:-1].astype(np.int64), np.diff(vptr.astype(np.int64))) + np.arange(int(ptr[-1]))
    out = torch.full((int(ptr[-1]) + 1,), -1, dtype=torch.int32, device="cuda")
    args = [_device(a) for a in (vptr, ptr, below.astype(np.uint32), np.append(cold, np.uint32(0)))]
    assert launch(args[0].data_ptr(), vptr.size - 1, args[1].data_ptr(), args[2].data_ptr(), args[3].data_ptr(), m,
                  out.data_ptr(), None) == 0
    torch.cuda.synchronize()
    got = out.cpu().numpy().view(np.uint32)
    assert np.array_equal(got[:-1], want.astype(np.uint32)) and got[-1] == 0xffffffff
