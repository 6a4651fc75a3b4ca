"""Child process of test_workspace_host.py: calls the library on a stand-in for the HIP runtime.  argv: the built stub, the
library, a JSON list of steps; prints a JSON list with what the runtime was asked for in every step."""
import ctypes as C
import json
import sys
import threading

stub = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
lib = C.CDLL(sys.argv[2])
lib.gz_gemm.argtypes = [C.c_int] + [C.c_void_p] * 4 + [C.c_int64] * 3 + [C.c_int] * 2 + [C.c_double] * 2 + [C.c_int] * 2 + [C.c_void_p]
lib.gz_gemm_static_scratch.argtypes = lib.gz_gemm.argtypes
lib.gz_last_error.restype = C.c_char_p
stub.stub_take.restype = C.c_char_p
stub.stub_capture.argtypes = [C.c_void_p]
A, B, D = 1 << 40, 2 << 40, 3 << 40   # never read: nothing runs


def gemm(types, m, n, k, la=0, lb=1, rung=-1, variant=0, stream=0, entry="gz_gemm"):
    st = getattr(lib, entry)(types, A, B, None, D, m, n, k, la, lb, 1.0, 0.0, rung, variant, stream)
    return [st, lib.gz_last_error().decode() if st else ""]


out = []
for step in json.loads(sys.argv[3]):
    what, args = step[0], step[1:]
    result = None
    if what == "gemm":
        result = gemm(**args[0])
    elif what == "other_thread":
        def work():
            global result
            result = gemm(**args[0])
        t = threading.Thread(target=work)
        t.start()
        t.join()
    else:
        getattr(stub, what)(*args)
    events = [line.split(" ", 3) for line in stub.stub_take().decode().splitlines()]
    out.append({"result": result, "events": [[e[0], int(e[1]), int(e[2]), e[3]] for e in events]})
print(json.dumps(out))
