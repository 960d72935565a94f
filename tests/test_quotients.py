"""The kernels' quotients by a corrected product: the bits of the IEEE division
for every binary32 argument (a quotient in binary64 rounded to binary32 is the
correctly rounded one: no quotient here lies within 2^-50 of a midpoint)."""

import ctypes as ct

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

CHUNK = 1 << 26


def _quotients(x, count):
    from hexdyn.lib import lib

    q = torch.full_like(x, -1.0)
    rc = lib().hexdyn_quotient(ct.c_void_p(x.data_ptr()), ct.c_void_p(q.data_ptr()), ct.c_int64(x.numel()),
                               ct.c_int(count), ct.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    return q


@pytest.mark.parametrize("count", [0, 3, 4, 5, 6, 7])
def test_every_argument(count):
    print(f"[gpu] quotients, {'1 / x' if count == 0 else f'x / {count}'}", flush=True)
    differ = torch.zeros((), dtype=torch.int64, device="cuda")
    for first in range(-(1 << 31), 1 << 31, CHUNK):
        x = torch.arange(first, first + CHUNK, device="cuda").to(torch.int32).view(torch.float32)
        want = (1.0 / x.double() if count == 0 else x.double() / count).float()
        got = _quotients(x, count)
        same = (want.view(torch.int32) == got.view(torch.int32)) | (want.isnan() & got.isnan())
        differ += (~same).sum()
    assert differ.item() == 0


def test_refusals():
    from hexdyn.lib import lib

    x = torch.ones(4, device="cuda")
    p = ct.c_void_p(x.data_ptr())
    for n, count in ((-1, 0), (4, 1), (4, 2), (4, 8), (4, -3)):
        assert lib().hexdyn_quotient(p, p, ct.c_int64(n), ct.c_int(count), None) != 0
    assert lib().hexdyn_quotient(None, p, ct.c_int64(4), ct.c_int(0), None) != 0
    assert lib().hexdyn_quotient(None, None, ct.c_int64(0), ct.c_int(0), None) == 0
