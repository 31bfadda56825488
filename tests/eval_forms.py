"""One evaluation pass chain called directly, in every input and output form
(the minimizers' trial points, signed and Newton forms have no entry point of
their own): the library's internal descriptor and the calls behind the C ABI."""
import ctypes as C
import os

import numpy as np

from tests.test_gpu_plane_fp64 import LAT

KINDS = {"wt": (0, 3), "wt4": (1, 4), "wgc": (2, 8), "spin": (3, 5), "spin4": (4, 7)}   # number, fields
IN_RHO, IN_PHI = 0, 1
OUT_POT, OUT_SIGNED, OUT_NEWTON = 0, 1, 2
NSUM = 11


class ReqDesc(C.Structure):   # as csrc/ofd_internal.h; the host-side test compares the layouts
    _fields_ = ([(n, C.c_void_p) for n in "u v bvec w vion out sums wgck wtk fin work".split()] +
                [(n, C.c_double) for n in "ca cb s1 s2 mu0 eps inv_eps".split()] + [("rb", C.c_double * 9)] +
                [(n, C.c_double) for n in "lam mu alpha beta rhoS coef tkf".split()] +
                [("opt_sqrt", C.c_int), ("pad", C.c_int)] + [(n, C.c_void_p) for n in "u2 v2 out2".split()] +
                [(n, C.c_double) for n in "ca2 cb2 s1b s2b mu0b".split()] +
                [("lsda", C.c_int), ("newton_ch", C.c_int), ("wtk32", C.c_void_p), ("hfin", C.c_void_p)])


PLAN_BYTES = 4096   # room for a ShapePlan


class Evaluator:
    """The passes of one grid and kind, with the environment's switches as they are now."""

    def __init__(self, grid, kind):
        import profess_amd
        from profess_amd.devmem import DeviceArray, hip
        self.L, self.hip, self.Dev = profess_amd.lib(), hip(), DeviceArray
        self.grid, self.kind = grid, kind
        n1, n2, n3 = grid
        self.shape, self.nc, self.rows = (n3, n2, n1), (n1 // 2 + 1) * n2 * n3, n2 * n3
        self.plan, err = C.create_string_buffer(PLAN_BYTES), C.create_string_buffer(64)
        init = self.L._ZN3ofd15shape_plan_initEPNS_9ShapePlanEiiiPNSt7__cxx1112basic_stringIcSt11char_traitsIcESaIcEEE
        assert init(self.plan, n1, n2, n3, err) == 0
        lat = LAT * (0.24 * np.array(grid))[None, :]
        self.rb = (2.0 * np.pi * np.linalg.inv(lat).T).ravel()

    def run(self, reqs, inmode, outmode):
        """reqs: dicts of host arrays (u, v, b, w, vion, wtk or wgck and with two
        channels u2, v2) and numbers, by the descriptor's names. One launch set;
        returns (out or [out, out2], sums) of each."""
        L, Dev, keep, outs = self.L, self.Dev, [], []
        descs = (ReqDesc * len(reqs))()
        for D, q in zip(descs, reqs):
            D.rb = (C.c_double * 9)(*self.rb)
            D.opt_sqrt, D.lsda, D.lam, D.mu, D.rhoS = 1, 2, 1.0, 1.0, 0.027
            for k, v in q.items():
                if isinstance(v, np.ndarray):
                    keep.append(Dev.from_host(v))
                    v = keep[-1].ptr
                setattr(D, k, v)
            buf = dict(out=Dev(self.shape), sums=Dev((self.rows * NSUM,)), fin=Dev((NSUM,)),
                       work=Dev((2 * KINDS[self.kind][1] * self.nc,)))
            if self.kind.startswith("spin"):
                buf["out2"] = Dev(self.shape)
            for k, v in buf.items():
                setattr(D, k, v.ptr)
            outs.append(buf)
        raw = np.frombuffer(bytes(descs), dtype=np.float64)   # copied as bytes
        dd = Dev.from_host(raw)
        k = KINDS[self.kind][0]
        run_eval = L._ZN3ofd8run_evalERKNS_9ShapePlanEiiiiPKNS_7ReqDescEiP12ihipStream_t
        fin = L._ZN3ofd12run_finalizeERKNS_9ShapePlanEiiPKNS_7ReqDescEiPdP12ihipStream_t
        assert run_eval(self.plan, k, inmode, outmode, 0, C.c_void_p(dd.ptr), len(reqs), None) == 0
        assert fin(self.plan, k, 0, C.c_void_p(dd.ptr), len(reqs), None, None) == 0
        assert self.hip.hipDeviceSynchronize() == 0
        return [([b[k].download() for k in ("out", "out2") if k in b], b["fin"].download()) for b in outs]


def environment(monkeypatch, generic):
    monkeypatch.setenv("OFD_GENERIC", "1" if generic else "0")
    assert "OFD_NO_PLANE" not in os.environ
