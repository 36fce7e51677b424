"""Rows past what one launch takes: the second launch starts where the first
ended. (The smallest tensors there are: a norm of 33.6 million rows of 257, in
place, and the positions of a layer step of 4 wide, 8.4 million.)"""
import pytest

from test_gpu_layer_launch import EPS, THETA, _inputs, _singles

pytestmark = pytest.mark.gpu


def test_norm(gpu):
    import torch
    rows, n = 2 ** 25 + 5, 257          # two rows a block of 256: 2^24 blocks are 2^32 threads
    if torch.cuda.mem_get_info()[0] < rows * n * 4 * 1.2:
        pytest.skip("needs 41 GB")
    x = torch.empty((rows, n), device="cuda")
    for part in x.split(2 ** 22):
        part.normal_()
    some = torch.tensor([0, 1, 7, 2 ** 24, 2 ** 25 - 4, 2 ** 25 - 3, 2 ** 25 - 2, 2 ** 25 - 1, 2 ** 25, rows - 2, rows - 1], device="cuda")
    ref = gpu.norm(x[some], 1e-5)
    mean = x[some].double().mean(1, keepdim=True)
    gpu.norm(x, 1e-5, out=x)
    assert torch.equal(x[some], ref)
    assert all(abs(part.double().mean()) < 1e-3 and abs(part[:, :8].float().std() - 1) < 0.01 for part in x.split(2 ** 23)[:-1])
    assert mean.abs().max() > 0.01      # (rows whose mean was not 0 before)
    del x
    torch.cuda.empty_cache()


def test_layer_step_goes_by_its_five_launches(gpu):
    import torch
    T = 2 ** 23
    a = _inputs(T, 4, 4, 1, 1, torch.bfloat16, 3)
    got = gpu.layer_nongemm_step(eps=EPS, n_dims=128, freq_base=THETA, **a)
    ref = _singles(gpu, a)
    for n in ref:
        assert torch.equal(got[n], ref[n]), n
    del got, ref, a
    torch.cuda.empty_cache()
