"""A unary set from host memory reaches the device whenever its upload runs.

A single instance's unary of 1 MiB and more waits in page-locked memory and is uploaded
beside the lattice builds (smaller ones, and those of several instances, wait in pageable
memory).  Whatever comes between setting it and the inference, the result has the bits of
an inference from the same unary in device memory.
"""
import ctypes

import numpy as np
import pytest
import torch

from pydensecrf_amd import capi
from tests.helpers import image_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H", [(120, 104), (120, 105), (333, 257)])  # 1 MiB - 4 KiB, over it, staged downloads
@pytest.mark.parametrize("order", ["before", "after", "between", "twice", "instance", "released", "abandoned"])
def test_upload_orders(W, H, order):
    L = 21
    img, U, _ = image_case(W, H, L, seed=7)
    other = np.ascontiguousarray(U[::-1]) + np.float32(1)
    ref = capi.Model.create_2d(W, H, L)  # (also: the process has used the device)
    ref.add_gaussian(3.0, 3.0, 3.0)
    ref.add_bilateral(40.0, 40.0, 13.0, 13.0, 13.0, img, 10.0)
    Ud = torch.from_numpy(np.ascontiguousarray(U.T)).cuda()
    want = torch.empty_like(Ud)
    torch.cuda.synchronize()
    ref.inference_device(2, want.data_ptr(), Ud.data_ptr())
    torch.cuda.synchronize()

    m = capi.Model.create_2d(W, H, L)
    if order in ("before", "released"):
        m.set_unary(U)
    elif order in ("twice", "instance"):
        m.set_unary(other)
    elif order == "abandoned":  # a model that goes with its upload under way; the next takes its buffer
        a = capi.Model.create_2d(W, H, L)
        a.set_unary(other)
        a.add_gaussian(3.0, 3.0, 3.0)
        del a
        m.set_unary(U)
    if order == "released":
        capi.check(capi.lib().dcrf_release_cached_memory(ctypes.byref(ctypes.c_size_t(0))))
    m.add_gaussian(3.0, 3.0, 3.0)
    if order in ("between", "twice"):
        m.set_unary(U)
    m.add_bilateral(40.0, 40.0, 13.0, 13.0, 13.0, img, 10.0)
    if order == "after":
        m.set_unary(U)
    elif order == "instance":
        m.set_unary_instance(0, U)
    for _ in range(2):  # the unary stays for later inferences
        got = np.ascontiguousarray(m.inference(2).T)
        assert np.array_equal(got.view(np.int32), want.cpu().numpy().view(np.int32))
    m.set_unary(other)  # and a later one takes its place
    assert not np.array_equal(np.ascontiguousarray(m.inference(2).T), got)
