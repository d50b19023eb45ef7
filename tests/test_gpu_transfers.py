"""Fields between host arrays and the device: chunks of 512 KiB through pinned
buffers, converted on the GPU.  Every value must arrive as the plain formula
gives it (FP32 states hold float32(v - offset) and give back that plus the
offset in FP64), at the edges of a chunk, across planes and with one, two and
four copying threads."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def S():
    import swalbe
    if swalbe.device_count() < 1:
        pytest.skip("no GPU")
    return swalbe


# 65536 doubles (131072 floats) fill a chunk; 1048576 doubles are 8 MiB (four threads)
SHAPES = [(1, 1), (7, 5), (512, 256), (513, 256), (511, 257), (1024, 1025), (1153, 911)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: f"{s[0]}x{s[1]}")
@pytest.mark.parametrize("host", [np.float64, np.float32], ids=["h64", "h32"])
@pytest.mark.parametrize("T", [np.float64, np.float32], ids=["d64", "d32"])
def test_fields_cross_as_the_formula_says(S, shape, host, T):
    Lx, Ly = shape
    print(f"[transfer] {shape} host {host.__name__} device {T.__name__}", flush=True)
    rng = np.random.default_rng(Lx * Ly)
    st = S.HipState(Lx, Ly, T=T)
    href, g = 0.7, 0.01
    st.set_reference_height(href, g)
    h32 = float(np.float32(href))
    R = np.array([np.float32(href * (1 - (5 / 6) * g * href))]
                 + [np.float32((1 / 9) * href * (1.5 * g * href))] * 4
                 + [np.float32((1 / 36) * href * (1.5 * g * href))] * 4, dtype=np.float64)
    for name, off in (("height", h32), ("velx", 0.0), ("feq", R)):
        if name == "feq" and Lx * Ly > 600_000:
            continue  # nine planes: sizes up to a few chunks a plane
        full = shape + ((9,) if name == "feq" else ())
        a = np.asfortranarray(0.7 + 0.3 * rng.standard_normal(full)).astype(host, order="F")
        st.set(name, a)
        want = a.astype(np.float64)
        if T is np.float32:
            want = np.float32(want - off).astype(np.float64) + off
        assert np.array_equal(st.get(name, np.float64), want), name
        assert np.array_equal(st.get(name, np.float32), want.astype(np.float32)), name
    st.close()


def test_raw_round_trip_keeps_every_bit(S):
    """Stored planes (checkpoints) cross unconverted: any bit pattern."""
    from swalbe import _lib
    L = _lib.lib()
    for T, U in ((np.float64, np.uint64), (np.float32, np.uint32)):
        st = S.HipState(300, 501, T=T)
        bits = np.random.default_rng(2).integers(0, np.iinfo(U).max, 9 * 300 * 501, dtype=U)
        _lib.check(L.swalbe_upload_raw(st.handle, 2, bits.ctypes.data, bits.nbytes))
        out = np.zeros_like(bits)
        _lib.check(L.swalbe_download_raw(st.handle, 2, out.ctypes.data, out.nbytes))
        assert np.array_equal(out, bits)
        st.close()


def test_new_reference_height_moves_the_encoding_only(S):
    """set_reference_height re-encodes in place: plain values stay to FP32 rounding of the
    deviation, and going there and back equals float32 arithmetic on the host."""
    h = np.asfortranarray(1.0 + 0.01 * np.random.default_rng(3).standard_normal((130, 70)))
    st = S.HipState(130, 70, T=np.float32)
    st.height = h
    d1 = np.float32(h - 1.0).astype(np.float64)
    st.set_reference_height(0.25)
    d2 = np.float32((d1 + 1.0) - 0.25).astype(np.float64)
    assert np.array_equal(st.get("height", np.float64), d2 + 0.25)
    st.close()


def test_line_fields_and_threads(S):
    """1D fields, and eight threads moving their own films at once."""
    import threading
    bad = []

    def work(k):
        try:
            rng = np.random.default_rng(k)
            st = S.HipState1D(40_000 + k, T=np.float64 if k % 2 else np.float32)
            for _ in range(5):
                a = rng.standard_normal((40_000 + k, 3))
                st.set("feq", np.asfortranarray(a))
                if not np.array_equal(st.get("feq", np.float64), a.astype(st.T).astype(float)):
                    bad.append(k)
            st.close()
        except Exception as e:  # reported below, in the test's own thread
            bad.append(e)
    ts = [threading.Thread(target=work, args=(k,)) for k in range(8)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad, bad
