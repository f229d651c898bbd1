"""CPU checks of Operation objects that come from elsewhere."""
import base64
import pickle
import types

import numpy as np

from quaru_amd import Register, _lib
from quaru_amd import operation as ops

# [not_(1), Operation.controlled([0, 2], X, [1], control_values=[True, False])]
# pickled when an Operation had no slot for the register's call
OLD = base64.b64decode(
    b"gASVzQEAAAAAAABdlCiME3F1YXJ1X2FtZC5vcGVyYXRpb26UjAlPcGVyYXRpb26Uk5QpgZROfZQojAdfbWF0cml4"
    b"lIwWbnVtcHkuX2NvcmUubXVsdGlhcnJheZSMDF9yZWNvbnN0cnVjdJSTlIwFbnVtcHmUjAduZGFycmF5lJOUSwCF"
    b"lEMBYpSHlFKUKEsBSwJLAoaUaAqMBWR0eXBllJOUjANjMTaUiYiHlFKUKEsDjAE8lE5OTkr/////Sv////9LAHSU"
    b"YolDQAAAAAAAAAAAAAAAAAAAAAAAAAAAAADwPwAAAAAAAAAAAAAAAAAA8D8AAAAAAAAAAAAAAAAAAAAAAAAAAAAA"
    b"AACUdJRijAhfdGFyZ2V0c5RdlEsBYYwJX2NvbnRyb2xzlF2UjAZfY3ZhbHOUTowGX2xhYmVslIwDbm90lHWGlGJo"
    b"AymBlE59lChoBmgJaAxLAIWUaA6HlFKUKEsBSwJLAoaUaBaJQ0AAAAAAAAAAAAAAAAAAAAAAAAAAAAAA8D8AAAAA"
    b"AAAAAAAAAAAAAPA/AAAAAAAAAAAAAAAAAAAAAAAAAAAAAAAAlHSUYmgbXZRLAWFoHV2UKEsASwJlaB9dlCiIiWVo"
    b"IIwAlHWGlGJlLg==")


def test_operations_pickled_without_a_call(monkeypatch):
    calls = []
    lib = types.SimpleNamespace(
        qs_apply=lambda h, *a: calls.append(("dense", a[-1])) or 0,
        qs_apply_controlled=lambda h, *a: calls.append(("controlled", a[-1])) or 0)
    monkeypatch.setattr(_lib, "load", lambda: lib)
    r = Register.__new__(Register)
    r._h = None
    for op in pickle.loads(OLD):
        r.apply(op)
    assert calls == [("dense", 1), ("controlled", 1)]
    a, b = pickle.loads(OLD)
    assert a == ops.not_(1)
    assert b.control_values == [True, False] and np.array_equal(b.active_matrix, a.matrix())
