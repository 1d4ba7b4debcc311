"""Which kernels calls of the C ABI launch, without a GPU: loads libsbq.so over
the launch recorder (launch_trace.cpp) and runs calls on made-up device
addresses, which host code never reads.

    dispatch.py RECORDER LIBRARY < calls > traces

stdin: a JSON list of calls, each a dict of plain values (see call()); stdout:
for each, {"rc": status, "launches": [[kernel, grid xyz, block xyz, LDS], ...]}
with demangled kernel names.  A process of its own: the recorder replaces the
HIP runtime for the whole process."""
import ctypes
import json
import subprocess
import sys

DT = {"f32": 0, "f16": 1, "bf16": 2}
ESIZE = {"f32": 4, "f16": 2, "bf16": 2}


def call(L, c):
    """Status of one call.  op: the entry point without its prefix; M, N, K, x
    (dtype), y (dtype, default f32); ws: "full" (sbq_linear_workspace_bytes),
    "base" (sbq_w8_workspace_bytes / sbq_w8a8_workspace_bytes), a number of
    base workspaces, or none; off: elements x starts beyond a 16-byte boundary;
    pad: elements added to x's row stride; count: linears of a grouped call;
    colsum: with column sums (repack_w8)."""
    P = ctypes.c_void_p
    at = lambda i: P((i + 1) << 40)  # noqa: E731
    op, M, N, K = c["op"], c.get("M", 0), c["N"], c.get("K", 0)
    x, y = c.get("x", "f32"), c.get("y", "f32")
    if op == "repack_w8":
        return L.sbq_repack_w8(at(0), N, K, K, at(1), at(4) if c.get("colsum") else None, None)
    if op == "argmax_rows":
        return L.sbq_argmax_rows(at(0), M, N, N, at(1), None)
    if op == "quantize_per_channel":
        return L.sbq_quantize_per_channel(at(0), DT[x], N, K, K, at(1), K, at(2), None)
    dyn = "w8a8" in op
    xp = P(at(0).value + c.get("off", 0) * ESIZE[x])
    ldx = K + c.get("pad", 0)
    base = L.sbq_w8a8_workspace_bytes(M, K) if dyn else L.sbq_w8_workspace_bytes(M, K, DT[x])
    ws = c.get("ws")
    nws = {None: 0, "base": base, "full": L.sbq_linear_workspace_bytes(M, N, K, DT[x], int(dyn))}.get(ws)
    if nws is None:
        nws = int(ws) * base
    wsp = at(6) if nws else None
    cs = (at(4),) if dyn and "token" not in op else ()
    head = (xp, DT[x], M, K, ldx, at(1), at(2)) + cs
    if op in ("linear_w8", "linear_w8a8", "linear_w8a8_token"):
        acc = (None,) if dyn else ()
        return getattr(L, "sbq_" + op)(*head, at(3), N, at(5), DT[y], N, *acc, wsp, nws, None)
    if op in ("linear_w8_parts", "linear_w8a8_parts"):
        return getattr(L, "sbq_" + op)(*head, at(3), N, at(5), DT[y], at(7), wsp, nws, None)
    if op in ("linear_w8_argmax", "linear_w8a8_argmax"):
        return getattr(L, "sbq_" + op)(*head, at(3), N, at(5), N, at(8), wsp, nws, at(9), None)
    if op in ("linear_w8_grouped", "linear_w8a8_grouped"):
        n = c.get("count", 2)
        ptrs = lambda i: (P * n)(*[at(i).value + (j << 36) for j in range(n)])  # noqa: E731
        longs = lambda v: (ctypes.c_int64 * n)(*[v] * n)  # noqa: E731
        xs = (P * n)(*[xp.value + (j << 36) for j in range(n)])
        args = (n, xs, longs(ldx), DT[x], M, K, ptrs(1), ptrs(2))
        tail = (ptrs(3), longs(N), ptrs(5), longs(N), DT[y])
        if dyn:
            return L.sbq_linear_w8a8_grouped(*args, ptrs(4), *tail, wsp, nws, None)
        return L.sbq_linear_w8_grouped(*args, *tail, None)
    raise ValueError(op)


def main():
    rec = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
    L = ctypes.CDLL(sys.argv[2])
    sys.path.insert(0, sys.argv[3])
    from _lib import SIGNATURES

    for name, (res, args) in SIGNATURES.items():
        if hasattr(L, name):
            f = getattr(L, name)
            f.restype, f.argtypes = res, args
    out, mangled = [], []
    buf, dims = ctypes.create_string_buffer(4096), (ctypes.c_int64 * 7)()
    for c in json.load(sys.stdin):
        rec.trace_reset()
        rc = call(L, c)
        launches = []
        for i in range(rec.trace_count()):
            rec.trace_get(i, buf, ctypes.c_size_t(len(buf)), dims)
            mangled.append(buf.value.decode())
            launches.append([len(mangled) - 1, list(dims)[0:3], list(dims)[3:6], dims[6]])
        out.append({"rc": rc, "launches": launches})
    names = subprocess.run(["c++filt"], input="\n".join(mangled), capture_output=True, text=True).stdout.split("\n")
    for o in out:
        for ln in o["launches"]:
            ln[0] = names[ln[0]].removeprefix("void ").removeprefix("sbq::").split("(")[0]
    json.dump(out, sys.stdout)


if __name__ == "__main__":
    main()
