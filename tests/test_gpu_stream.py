"""Calls without a stream argument run on torch's current stream: the default
one, a stream made current, and the default again."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
import datagen as dg
import nnops_amd as na
from nnops_amd import ops
from gpu_util import dev, host, announce

pytestmark = pytest.mark.gpu


def test_current_stream():
    import torch
    announce("current stream")
    M, K, N = 3, 256, 64
    a, w = dg.act_s8(1, (M, K)), dg.ints(2, (N, K), -127, 127)
    da, dw = dev(a), dev(w)
    want = oracle.gemm_i8(a, w, trans_b=True)
    side = torch.cuda.Stream()
    for stream in (torch.cuda.default_stream(), side, torch.cuda.default_stream()):
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            assert (ops._stream_ptr(None) or 0) == stream.cuda_stream
            c = torch.zeros((M, N), dtype=torch.int32, device="cuda")
            na.gemm_i8(da, dw, c, trans_b=True)
            stream.synchronize()
        assert np.array_equal(host(c), want)
    assert (ops._stream_ptr(side) or 0) == side.cuda_stream


def test_current_stream_without_the_private_name(monkeypatch):
    """A torch whose raw stream lookup has another name: the Stream object's
    handle."""
    import torch
    announce("current stream, public names only")
    monkeypatch.setattr(ops, "_RAW_STREAM", None)
    monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream")
    side = torch.cuda.Stream()
    for stream in (side, torch.cuda.default_stream()):
        with torch.cuda.stream(stream):
            assert (ops._stream_ptr(None) or 0) == stream.cuda_stream
