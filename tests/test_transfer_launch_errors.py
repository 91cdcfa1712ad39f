"""Host transfers report a refused launch.  On the CPU, on a stand-in for the HIP
runtime whose next launch can be made to fail.  Neither the copies around the
repitch kernel nor a stream synchronisation return a refused launch's error, and a
transfer must not clear one that an earlier call left."""
from tests import fakehip

CHILD = r"""
C = L.Context((9, 8, 7), (0.1, 0.1, 0.1))
a = np.ones(C.shape)
C.upload(L.FIELD_T0, a)
C.download(L.FIELD_T0)
assert fake.fake_launches() >= 2  # pageable memory takes the repitch kernel
for call in (lambda: C.upload(L.FIELD_T0, a), lambda: C.download(L.FIELD_T0)):
    fake.fake_set(1, 0)
    try:
        call()
    except L.PPSError as e:
        assert "repitch" in str(e), e
    else:
        sys.exit("a refused repitch launch was not reported")
    fake.fake_set(0, 0)
    fake.hipGetLastError()
for attr_fails in (0, 1):
    # an earlier call's refused launch stays pending over a transfer
    fake.fake_set(1, 0)
    C.fill(L.FIELD_T0, 1.0)
    fake.fake_set(0, attr_fails)
    C.upload(L.FIELD_T0, a)
    if fake.hipGetLastError() == 0:
        sys.exit("the transfer cleared an error that an earlier launch had left")
    # and a transfer's own tolerated failure leaves none behind
    C.upload(L.FIELD_T0, a)
    if fake.hipGetLastError() != 0:
        sys.exit("the transfer left an error of its own")
print("ok")
"""


def test_refused_launches_are_reported(tmp_path):
    assert fakehip.run(tmp_path, CHILD).strip() == "ok"
