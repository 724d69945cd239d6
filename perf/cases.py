"""The workloads that the library's speed is judged on.

A case is a dict of plain values.  `prepare` makes what a program holds before
the call (integer arrays resident on the GPU, a prepared batch, or host
buffers), `run` makes one pass through the C API as a program calls it and
returns the whole results: arithmetic results are exported into a device
tensor, a call on host buffers returns host arrays.

The kinds:
  powm   out = base^exp mod m; "shared" keys have one modulus and exponent
  add, sub, mul, sqr, div, mod, divmod
  bytes  big-endian byte strings in host memory imported and exported again
  crt    CRT decryption under one resident key, host buffers to host buffers
  batch  one prepared launch over instances of mixed modulus sizes
"""
import math

import numpy as np
import torch

import xmp_amd
from xmp_amd import ext, inputs


def listed():
    return [
        # the headline: private-key operations in bulk
        {"name": "powm_2048", "kind": "powm", "bits": 2048, "exp_bits": 2048, "count": 65536, "shared": False},
        # CRT halves or 1024-bit groups, a batch that only just fills the GPU
        {"name": "powm_1024_small", "kind": "powm", "bits": 1024, "exp_bits": 1024, "count": 4096, "shared": False},
        # signature verification: exponent 65537 under many keys
        {"name": "powm_2048_verify", "kind": "powm", "bits": 2048, "exp_bits": 32, "count": 16384, "shared": False},
        # key agreement in one 3072-bit group, short exponents, a ragged batch
        {"name": "powm_3072_group", "kind": "powm", "bits": 3072, "exp_bits": 256, "count": 1000, "shared": True},
        # a service's mixed queue in one launch, 512- to 8192-bit moduli
        {"name": "batch_mixed", "kind": "batch", "count": 16384},
        # CRT decryption of a request batch, host to host
        {"name": "crt_decrypt", "kind": "crt", "bits": 2048, "count": 4096},
        # streaming sums
        {"name": "add_2048", "kind": "add", "bits": 2048, "bits_b": 2048, "count": 1048576},
        # key-size products in bulk
        {"name": "mul_2048", "kind": "mul", "bits": 2048, "bits_b": 2048, "count": 1048576},
        # long products
        {"name": "mul_32768", "kind": "mul", "bits": 32768, "bits_b": 32768, "count": 4096},
        # reduction of double-length products, quotient and remainder
        {"name": "divmod_4096", "kind": "divmod", "bits": 4096, "bits_b": 2048, "count": 65536, "shared": False},
        # the smallest calls: a few hundred odd-sized reductions
        {"name": "mod_1568_few", "kind": "mod", "bits": 1568, "bits_b": 1056, "count": 300, "shared": False},
        # messages and signatures as byte strings in host memory
        {"name": "bytes_2048", "kind": "bytes", "bits": 2048, "count": 16384},
    ]


# No drawn case costs more than the listed batches: 32-bit multiply-adds of an
# exponentiation, of a product or division, and bytes moved.
_POWM_MACS = 65536 * 2048 * 1.2 * (2 * 64 * 64 + 64)
_POWM_CHAIN = 6144 * 1.2 * 192 * 192   # one instance's serial work: the largest class that one draw may hold alone
_MUL_MACS = 4096 * 1024.0 ** 2
_DIV_MACS = 65536 * 64.0 * 64.0 * 4
_BYTES = 1048576 * 768.0


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))


def _count(rng, cap):
    """A batch size: a library of batched calls is called for some instances at a time."""
    cap = max(1, int(cap))
    return _log_int(rng, min(16, cap), cap)


def _bits(rng, lo, hi):
    """A size in whole limbs; half of them the round sizes that keys have."""
    if rng.random() < 0.5:
        usual = [b for b in (64, 128, 256, 512, 768, 1024, 1536, 2048, 3072, 4096, 6144, 8192, 16384, 32768) if lo <= b <= hi]
        return rng.choice(usual)
    return max(lo, min(hi, 32 * max(1, _log_int(rng, lo, hi) // 32)))


def draw(rng):
    kind = rng.choice(["powm", "powm", "powm", "powm", "mul", "mul", "sqr", "divmod", "div", "mod", "add", "sub",
                       "bytes", "crt"])
    if kind == "powm":
        bits = _bits(rng, 256, 6144)
        n = bits // 32
        exp_bits = rng.choice([32, 256, bits, bits])
        macs = exp_bits * 1.2 * (2 * n * n + n)
        cap = int(min(65536, max(1, _POWM_MACS / macs)))
        if exp_bits * 1.2 * n * n > _POWM_CHAIN / 8:
            cap = min(cap, 2048)
        return {"kind": kind, "bits": bits, "exp_bits": exp_bits, "count": _count(rng, cap),
                "shared": rng.random() < 0.25}
    if kind in ("mul", "sqr"):
        bits = _bits(rng, 128, 65536)
        bits_b = bits if kind == "sqr" or rng.random() < 0.6 else _bits(rng, 64, bits)
        limbs = bits // 32, bits_b // 32
        cap = min(1048576, _MUL_MACS / (limbs[0] * limbs[1]), _BYTES / (8.0 * (limbs[0] + limbs[1])))
        return {"kind": kind, "bits": bits, "bits_b": bits_b, "count": _count(rng, cap)}
    if kind in ("div", "mod", "divmod"):
        bits_b = _bits(rng, 64, 8192)
        bits = min(32768, max(bits_b, 32 * int(bits_b * rng.choice([1.5, 2, 2, 3]) / 32)))
        limbs = bits // 32, bits_b // 32
        cap = min(524288, _DIV_MACS / (limbs[0] * limbs[1]), _BYTES / (8.0 * (limbs[0] + limbs[1])))
        return {"kind": kind, "bits": bits, "bits_b": bits_b, "count": _count(rng, cap),
                "shared": rng.random() < 0.25}
    if kind in ("add", "sub"):
        bits = _bits(rng, 64, 8192)
        bits_b = bits if rng.random() < 0.7 else _bits(rng, 64, bits)
        cap = min(4194304, _BYTES / (12.0 * (bits // 32)))
        return {"kind": kind, "bits": bits, "bits_b": bits_b, "count": _count(rng, cap)}
    if kind == "bytes":
        bits = _bits(rng, 256, 8192)
        return {"kind": kind, "bits": bits, "count": _count(rng, 16384 * 2048 // bits)}
    return {"kind": "crt", "bits": rng.choice([1024, 2048, 3072, 4096]), "count": _count(rng, 2048)}


# ---- inputs -----------------------------------------------------------------

_handle = None


def _h():
    """The program's handle, one for all of its calls."""
    global _handle
    if _handle is None:
        _handle = xmp_amd.Handle()
    return _handle


def _uniform(gen, count, bits):
    return torch.randint(-2 ** 31, 2 ** 31, (count, bits // 32), dtype=torch.int64, device="cuda",
                         generator=gen).to(torch.int32)


def _top_set(t):
    t[:, -1] |= -2 ** 31
    return t


def _odd(t):
    t[:, 0] |= 1
    return t


def _below(t):
    """Below any integer of the same length whose top bit is set."""
    t[:, -1] &= 2 ** 31 - 1
    return t


def _numbers(case, seed):
    """The operands of an arithmetic case, as (count, limbs) int32 tensors."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    kind, n = case["kind"], case["count"]
    if kind == "powm":
        keys = 1 if case["shared"] else n
        m = _odd(_top_set(_uniform(gen, keys, case["bits"])))
        b = _below(_uniform(gen, n, case["bits"]))
        if case["exp_bits"] == 32:
            e = torch.full((1, 1), 65537, dtype=torch.int32, device="cuda")
        else:
            e = _uniform(gen, n, case["exp_bits"])
        return b, e, m
    a = _uniform(gen, n, case["bits"])
    if kind == "sqr":
        return (a,)
    rows = 1 if case.get("shared") else n
    b = _uniform(gen, rows, case["bits_b"])
    if kind in ("div", "mod", "divmod"):
        b = _top_set(b)
    return a, b


def _load(t):
    """A device tensor of limbs as a resident integer array."""
    h = _h()
    x = h.integers(32 * t.shape[1], t.shape[0])
    xmp_amd.check(xmp_amd.lib().xmpIntegersImport(h.h, x.x, t.shape[1], -1, 4, 0, 0, t.data_ptr(), t.shape[0]),
                  "xmpIntegersImport")
    return x


def _results(bits, count):
    """A result array and the device tensor that it is exported into."""
    return _h().integers(bits, count), torch.empty((count, bits // 32), dtype=torch.int32, device="cuda")


class _Batch:
    """A prepared batch, released with the state that holds it."""

    def __init__(self, *args):
        self.batch = ext.Batch(*args)
        self.batch.prepare()

    def __del__(self):
        self.batch.close()


def _key(bits, seed):
    """One CRT key: the moduli, exponents and coefficients as host rows."""
    return ext.make_keys(1, bits, 2 * (seed % 1000003) + 1)


def prepare(case, seed):
    kind, n = case["kind"], case.get("count")
    if kind == "bytes":
        rng = np.random.Generator(np.random.PCG64(seed))
        src = rng.integers(0, 256, (n, case["bits"] // 8), dtype=np.uint8)
        return {"kind": kind, "src": src, "dst": np.zeros_like(src), "x": _h().integers(case["bits"], n),
                "count": n}
    if kind == "crt":
        bits = case["bits"]
        key = _key(bits, seed)
        rng = np.random.Generator(np.random.PCG64(seed))
        src = rng.integers(0, 2 ** 32, (n, bits // 32), dtype=np.uint32)
        src[:, -1] &= 0x3FFFFFFF   # below n
        h = _h()
        s = {"kind": kind, "src": src, "dst": np.zeros_like(src), "count": n,
             "key": {k: h.from_array(v) for k, v in key.items()}}
        for name, b in (("c", bits), ("r", bits // 2), ("mp", bits // 2), ("mq", bits // 2),
                        ("sp", bits + bits // 2 + 32), ("sq", bits + bits // 2 + 32), ("out", bits)):
            s[name] = h.integers(b, n)
        return s
    if kind == "batch":
        counts = inputs.mixed_counts(n, 777)   # the queue's make-up is the same for every seed
        arrays = []
        for j, (bits, cnt) in enumerate(zip(inputs.MIXED_SIZES, counts)):
            if cnt == 0:
                continue
            b, e, m = _numbers({"kind": "powm", "bits": bits, "exp_bits": bits, "count": cnt, "shared": False},
                               seed + 7919 * (j + 1))
            arrays.append((_results(bits, cnt), _load(b), _load(e), _load(m), cnt))
        outs = [a[0] for a in arrays]
        return {"kind": kind, "outs": outs,
                "batch": _Batch(_h(), [o[0] for o in outs], [a[1] for a in arrays], [a[2] for a in arrays],
                                [a[3] for a in arrays], [a[4] for a in arrays])}
    ops = [_load(t) for t in _numbers(case, seed)]
    sizes = {"powm": [case["bits"]], "add": [case["bits"]], "sub": [case["bits"]], "sqr": [2 * case["bits"]],
             "mul": [case["bits"] + case.get("bits_b", 0)], "div": [case["bits"]], "mod": [case.get("bits_b", 0)],
             "divmod": [case["bits"], case.get("bits_b", 0)]}[kind]
    return {"kind": kind, "ops": ops, "outs": [_results(b, n) for b in sizes], "count": n}


# ---- one pass ---------------------------------------------------------------


def _export(outs):
    h, L = _h(), xmp_amd.lib()
    for x, t in outs:
        xmp_amd.check(L.xmpIntegersExportAsync(h.h, t.data_ptr(), None, -1, 4, 0, 0, x.x, x.count),
                      "xmpIntegersExportAsync")
    return [t for _, t in outs]


_CALLS = {"powm": "xmpIntegersPowmAsync", "add": "xmpIntegersAddAsync", "sub": "xmpIntegersSubAsync",
          "mul": "xmpIntegersMulAsync", "sqr": "xmpIntegersSqrAsync", "div": "xmpIntegersDivAsync",
          "mod": "xmpIntegersModAsync", "divmod": "xmpIntegersDivModAsync"}


def run(state):
    h, L, kind = _h(), xmp_amd.lib(), state["kind"]
    if kind in _CALLS:
        args = [x.x for x, _ in state["outs"]] + [x.x for x in state["ops"]]
        xmp_amd.check(getattr(L, _CALLS[kind])(h.h, *args, state["count"]), _CALLS[kind])
        return _export(state["outs"])
    if kind == "batch":
        state["batch"].batch.launch_async()
        return _export(state["outs"])
    n = state["count"]
    if kind == "bytes":
        src, dst, x = state["src"], state["dst"], state["x"]
        xmp_amd.check(L.xmpIntegersImport(h.h, x.x, src.shape[1], 1, 1, 1, 0, src.ctypes.data, n), "import")
        xmp_amd.check(L.xmpIntegersExport(h.h, dst.ctypes.data, None, 1, 1, 1, 0, x.x, n), "export")
        return dst
    # crt: mp = c^dp mod p, mq = c^dq mod q, out = (mp cp + mq cq) mod n
    k, src, dst = state["key"], state["src"], state["dst"]
    x = {name: state[name].x for name in ("c", "r", "mp", "mq", "sp", "sq", "out")}
    ok = xmp_amd.check
    ok(L.xmpIntegersImportAsync(h.h, x["c"], src.shape[1], -1, 4, 0, 0, src.ctypes.data, n), "import")
    for prime, exp, half in (("p", "dp", "mp"), ("q", "dq", "mq")):
        ok(L.xmpIntegersModAsync(h.h, x["r"], x["c"], k[prime].x, n), "mod")
        ok(L.xmpIntegersPowmAsync(h.h, x[half], x["r"], k[exp].x, k[prime].x, n), "powm")
    ok(L.xmpIntegersMulAsync(h.h, x["sp"], x["mp"], k["cp"].x, n), "mul")
    ok(L.xmpIntegersMulAsync(h.h, x["sq"], x["mq"], k["cq"].x, n), "mul")
    ok(L.xmpIntegersAddAsync(h.h, x["sp"], x["sp"], x["sq"], n), "add")
    ok(L.xmpIntegersModAsync(h.h, x["out"], x["sp"], k["n"].x, n), "mod")
    ok(L.xmpIntegersExport(h.h, dst.ctypes.data, None, -1, 4, 0, 0, x["out"], n), "export")
    return dst


# ---- the work a pass cannot do without --------------------------------------


def _powm_work(bits, exp_bits, n):
    """Squarings and fixed-window products of 2 limbs^2 + limbs multiply-adds each, two operations a multiply-add."""
    limbs = bits // 32
    w = min(range(1, 9), key=lambda w: 2 ** w + -(-exp_bits // w))
    return 2.0 * n * (exp_bits + -(-exp_bits // w)) * (2 * limbs * limbs + limbs)


def work(case):
    kind, n = case["kind"], case.get("count")
    if kind == "batch":
        parts = [({"kind": "powm", "bits": b, "exp_bits": b, "count": n * w, "shared": False})
                 for b, w in zip(inputs.MIXED_SIZES, inputs.MIXED_WEIGHTS)]
        done = [work(p) for p in parts]
        return {"bytes": sum(d["bytes"] for d in done), "flops": sum(d["flops"] for d in done)}
    a = case["bits"] // 32
    if kind == "bytes":
        return {"bytes": 8.0 * a * n, "flops": 0.0}
    if kind == "crt":
        h = a // 2
        return {"bytes": 8.0 * a * n,
                "flops": 2 * _powm_work(16 * a, 16 * a, n) + 2.0 * n * (2 * h * h + 2 * a * h + (a + h) * h)}
    if kind == "powm":
        keys = 1 if case["shared"] else n
        e = case["exp_bits"] // 32 * (1 if case["exp_bits"] == 32 else n)
        return {"bytes": 4.0 * (2 * a * n + a * keys + e), "flops": _powm_work(case["bits"], case["exp_bits"], n)}
    b = case["bits_b"] // 32 if kind != "sqr" else 0
    rows = 1 if case.get("shared") else n
    if kind in ("add", "sub"):
        return {"bytes": 4.0 * n * (2 * a + b), "flops": 1.0 * n * a}
    if kind == "sqr":
        return {"bytes": 4.0 * n * 3 * a, "flops": 1.0 * n * a * (a + 1)}
    if kind == "mul":
        return {"bytes": 4.0 * n * 2 * (a + b), "flops": 2.0 * n * a * b}
    out = {"div": a, "mod": b, "divmod": a + b}[kind]
    return {"bytes": 4.0 * (n * (a + out) + rows * b), "flops": 2.0 * n * (a - b + 1) * b}


# ---- exact results ----------------------------------------------------------


def _ints(t):
    rows = t.cpu().numpy().astype("<i4") if isinstance(t, torch.Tensor) else t
    return [int.from_bytes(r.tobytes(), "little") for r in rows]


def _rows(values, bits):
    data = b"".join((v & (1 << bits) - 1).to_bytes(bits // 8, "little") for v in values)
    return np.frombuffer(data, "<i4").reshape(len(values), bits // 32)


def exact(case, seed):
    """The same results by Python's integers, where that takes seconds."""
    kind, n = case["kind"], case.get("count")
    if kind in ("batch", "crt"):
        return None
    if kind == "bytes":
        rng = np.random.Generator(np.random.PCG64(seed))
        return rng.integers(0, 256, (n, case["bits"] // 8), dtype=np.uint8)
    w = work(case)
    if w["flops"] > 2e10 or n > 300000:
        return None
    ops = [_ints(t) for t in _numbers(case, seed)]
    bits = case["bits"]
    if kind == "powm":
        b, e, m = ops
        return [_rows([pow(b[i], e[i % len(e)], m[i % len(m)]) for i in range(n)], bits)]
    if kind == "sqr":
        return [_rows([x * x for x in ops[0]], 2 * bits)]
    a, b = ops[0], ops[1] * (n // len(ops[1]))
    if kind == "add":
        return [_rows([x + y for x, y in zip(a, b)], bits)]
    if kind == "sub":
        return [_rows([x - y for x, y in zip(a, b)], bits)]
    if kind == "mul":
        return [_rows([x * y for x, y in zip(a, b)], bits + case["bits_b"])]
    both = [divmod(x, y) for x, y in zip(a, b)]
    q, r = _rows([x[0] for x in both], bits), _rows([x[1] for x in both], case["bits_b"])
    return {"div": [q], "mod": [r], "divmod": [q, r]}[kind]
