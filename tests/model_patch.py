"""Copies of a sam3.cpp model file with some of its F32 / F16 tensors replaced
(test helper)."""
import numpy as np

import oracle_lib as orc


def patched(src: str, dst: str, tensors: dict) -> None:
    """dst = src with the data of each named tensor replaced: an array of the tensor's size, or a number for all of it."""
    data = bytearray(open(src, "rb").read())
    records = orc.read_model_file(src)
    for name, value in tensors.items():
        dt, _, arr = records[name]
        assert dt in (0, 1), name
        new = np.broadcast_to(np.asarray(value, np.float32), arr.shape).astype(arr.dtype)
        # the record's name, then its data at the next multiple of 32
        at = data.index(name.encode(), 16)
        assert data.count(name.encode()) == 1, name
        at = (at + len(name) + 31) // 32 * 32
        assert data[at : at + arr.nbytes] == arr.tobytes(), name
        data[at : at + arr.nbytes] = new.tobytes()
    open(dst, "wb").write(data)
