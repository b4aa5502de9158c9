"""Autotuner for the engine's launch choices on the device at hand.

The reference makes one choice for every size (numpy.linalg.eigh per
instance, muspinsim/spinop.py:69, inside the loop of experiment.py:369).
Here the batch runs through different kernels depending on the Hilbert
dimension n and the number of instances of that dimension, and the best
choice is measured, not assumed:

  eigh          for each bucket n (and a ladder of batch sizes), the LDS
                Jacobi eigensolver (n <= 64) or MSP_EIGH_DC (one-wave Jacobi up
                to n = 16, Householder + divide and conquer above).
  timesum       the smallest n from which the FP64 time sum from a phase table
                on matrix cores (msp_timesum_mfma64) beats msp_timesum, and
                the smallest n from which the mixed-precision time sum (FP32
                matrix cores) beats the faster FP64 one on the same batch.
  max_chunk     instances per launch of the n = 192 divide-and-conquer path.

`tune()` times them with HIP events around the library calls and returns a
dict; `main()` writes it to JSON (muspinsim_amd/tuning.json by default),
which SpinEngine(tuning=...) reads at plan time.  Usage on the GPU:

    python -m muspinsim_amd.autotune [--out PATH] [--quick]
"""

import argparse
import json
import os
import time

HERE = os.path.dirname(os.path.abspath(__file__))
DEFAULT_PATH = os.path.join(HERE, "tuning.json")

EIGH_NS = (4, 8, 12, 16, 24, 32, 48, 64)
EIGH_BATCHES = (64, 256, 1024, 4096, 16384)
TIMESUM_NS = (16, 24, 32, 40, 48, 64, 72, 80, 96, 112, 128, 192, 256)


def _events_ms(fn, reps, before=None):
    """Best-of-reps milliseconds of fn, each after an untimed `before`."""
    import torch
    fn()                                   # warm up (kernel attributes, caches)
    torch.cuda.synchronize()
    a = torch.cuda.Event(enable_timing=True)
    b = torch.cuda.Event(enable_timing=True)
    best = float("inf")
    for _ in range(reps):
        if before is not None:
            before()
        a.record()
        fn()
        b.record()
        torch.cuda.synchronize()
        best = min(best, a.elapsed_time(b))
    return best


def _herm(n, batch, seed):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    X = torch.randn((batch, n, n), dtype=torch.complex128, device="cuda", generator=g)
    return (X + X.conj().transpose(1, 2).contiguous()) / 2


def time_eigh(lib, n, batch, method, reps=3):
    """Best-of-reps milliseconds of one msp_eigh call on random Hermitian
    matrices (the input is restored from a copy before every call)."""
    import torch
    from . import _native as N
    H0 = _herm(n, batch, 1000 + n)
    H = torch.empty_like(H0)
    E = torch.empty((batch, n), dtype=torch.float64, device="cuda")
    U = torch.empty_like(H0)
    info = torch.empty((batch,), dtype=torch.int32, device="cuda")
    wsb = lib.msp_eigh_workspace(n, batch, method)
    work = torch.empty((max(wsb, 8) // 8,), dtype=torch.float64, device="cuda")
    st = torch.cuda.current_stream().cuda_stream

    def call():
        H.copy_(H0)
        N.check(lib.msp_eigh(n, batch, H.data_ptr(), E.data_ptr(), U.data_ptr(), info.data_ptr(),
                             method, work.data_ptr(), wsb, st))

    copy_ms = _events_ms(lambda: H.copy_(H0), reps)
    return max(_events_ms(call, reps) - copy_ms, 1e-4)


def eigh_ladders(raw, tol=0.05):
    """{n: [[batch_min, method], ...]} from timings {"<n>x<batch>": {"jacobi_ms",
    "dc_ms"}}: the faster eigensolver from each batch size on, switching only
    when the other method is faster by more than `tol` (differences within the
    run-to-run noise keep the previous choice)."""
    by_n = {}
    for key, t in raw.items():
        n, batch = (int(x) for x in key.split("x"))
        by_n.setdefault(n, []).append((batch, t["jacobi_ms"], t["dc_ms"]))
    table = {}
    for n, rows in sorted(by_n.items()):
        ladder = []
        for batch, tj, td in sorted(rows):
            if not ladder:
                ladder.append([1, "jacobi" if tj <= td else "dc"])
                continue
            cur = ladder[-1][1]
            t_cur, t_other = (tj, td) if cur == "jacobi" else (td, tj)
            if t_other < t_cur * (1.0 - tol):
                ladder.append([batch, "dc" if cur == "jacobi" else "jacobi"])
        table[str(n)] = ladder
    return table


def tune_eigh(lib, ns=EIGH_NS, batches=EIGH_BATCHES, reps=3):
    """Eigensolver ladders per dimension (eigh_ladders) and the raw timings."""
    from . import _native as N
    raw = {}
    for n in ns:
        for batch in batches:
            tj = time_eigh(lib, n, batch, N.MSP_EIGH_JACOBI, reps)
            td = time_eigh(lib, n, batch, N.MSP_EIGH_DC, reps)
            raw[f"{n}x{batch}"] = {"jacobi_ms": tj, "dc_ms": td}
    return eigh_ladders(raw), raw


def tune_timesum(lib, ns=TIMESUM_NS, ntimes=2000, batch=256, reps=3, tol=0.1):
    """(first_table, first_mixed, raw): the smallest n (of ns) where
    msp_timesum_mfma64 is faster than msp_timesum and from which on it is never
    slower by more than `tol`, the same for the mixed-precision time sum against
    the faster of the two, and the timings of all three, with the caches filled
    with other data first: in a plan the weights come from HBM (n = 64, 256 x 2000
    times, msp_timesum 0.39 ms in a loop, 0.41 so, 0.43 in a plan; with the table
    0.38, 0.39, 0.38).  Up to n = MSP_TIMESUM_WAVE_N the first two are one kernel;
    only msp_timesum is timed there, which needs no phase table."""
    import torch
    from . import _native as N
    raw = {}
    st = torch.cuda.current_stream().cuda_stream
    t = torch.linspace(0, 10, ntimes, dtype=torch.float64, device="cuda")
    other = torch.empty((1 << 27,), dtype=torch.float64, device="cuda")    # 1 GiB

    def flush():
        other.fill_(1.0)

    for n in ns:
        E = torch.sort(torch.randn((batch, n), dtype=torch.float64, device="cuda") * 50, dim=1).values
        C = torch.randn((batch, n, n), dtype=torch.float64, device="cuda")
        C = ((C + C.transpose(1, 2)) / 2).contiguous()
        out = torch.empty((batch, ntimes), dtype=torch.float64, device="cuda")

        def table_ms(fn, workspace):
            ws = workspace(n, batch, ntimes)
            work = torch.empty((max(ws, 8) // 8,), dtype=torch.float64, device="cuda")
            return _events_ms(lambda: N.check(fn(n, batch, ntimes, E.data_ptr(), C.data_ptr(),
                                                 t.data_ptr(), None, out.data_ptr(),
                                                 work.data_ptr(), ws, st)), reps, flush)

        r = {"direct_ms": _events_ms(lambda: N.check(lib.msp_timesum(
            n, batch, ntimes, E.data_ptr(), C.data_ptr(), 1, t.data_ptr(), None, 0,
            out.data_ptr(), st)), reps, flush)}
        if n > N.MSP_TIMESUM_WAVE_N:
            r["table_ms"] = table_ms(lib.msp_timesum_mfma64, lib.msp_timesum_mfma64_workspace)
        r["mixed_ms"] = table_ms(lib.msp_timesum_mixed, lib.msp_timesum_mixed_workspace)
        raw[str(n)] = r
        del E, C, out
        torch.cuda.empty_cache()
    return timesum_thresholds(raw, tol) + (raw,)


def timesum_thresholds(raw, tol=0.1):
    """(first_table, first_mixed) from timings {"<n>": {"direct_ms", "table_ms"
    (absent where it is the same kernel), "mixed_ms"}}; a very large n when there
    is none."""
    def first(pair):
        best = 1 << 30
        for n in sorted((int(k) for k in raw), reverse=True):
            new, old = pair(raw[str(n)])
            if new > old * (1.0 + tol):
                break
            if new < old:
                best = n
        return best

    never = float("inf")
    return (first(lambda r: (r.get("table_ms", never), r["direct_ms"])),
            first(lambda r: (r["mixed_ms"], min(r.get("table_ms", never), r["direct_ms"]))))


def tune_chunk(candidates=(2048, 4096, 8192), nfields=40, nori=500):
    """Instances per launch for the n = 192 integral sweep: best of one
    timed execute per candidate on a 40-field slice of the sweep."""
    import torch
    from . import workloads as W
    from .engine import SpinEngine
    systems, batch = W.c2_alc_sweep(nfields=nfields, nori=nori)
    raw = {}
    for c in candidates:
        eng = SpinEngine("cuda:0", max_chunk=c, tuning=None)
        plan = eng.prepare(systems, batch)
        eng.execute(plan)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        eng.execute(plan)
        torch.cuda.synchronize()
        raw[str(c)] = (time.perf_counter() - t0) * 1e3
        del plan
        torch.cuda.empty_cache()
    return choose_chunk(raw), raw


def choose_chunk(raw, tol=0.02):
    """The largest candidate within `tol` of the fastest: larger chunks fill
    whole residency waves of the full sweep, which the slice does not show."""
    fastest = min(raw.values())
    return max(int(c) for c, ms in raw.items() if ms <= fastest * (1 + tol))


def tune(quick=False):
    import torch
    from . import _native as N
    lib = N.lib()
    reps = 2 if quick else 3
    batches = (64, 1024, 8192) if quick else EIGH_BATCHES
    eigh, eigh_raw = tune_eigh(lib, batches=batches, reps=reps)
    table_min, mixed_min, ts_raw = tune_timesum(lib, reps=reps)
    chunk, chunk_raw = tune_chunk() if not quick else (8192, {})
    return {
        "device": torch.cuda.get_device_properties(0).gcnArchName,
        "eigh": eigh,
        "mixed_timesum_min_n": mixed_min,
        "fp64_timesum_mfma_min_n": table_min,
        "max_chunk": chunk,
        "measured": {"eigh_ms": eigh_raw, "timesum_ms": ts_raw, "chunk_ms": chunk_raw},
    }


def load(path=DEFAULT_PATH):
    """The tuning dict at `path`, or None when there is none."""
    if not path or not os.path.exists(path):
        return None
    with open(path) as f:
        return json.load(f)


def eigh_method(tuning, n, batch):
    """MSP_EIGH_* for n instances of dimension n from a tuning dict (AUTO
    when the tuning has no entry for n)."""
    from . import _native as N
    if not tuning:
        return N.MSP_EIGH_AUTO
    ladder = tuning.get("eigh", {}).get(str(int(n)))
    if not ladder:
        return N.MSP_EIGH_AUTO
    choice = ladder[0][1]
    for bmin, m in ladder:
        if batch >= bmin:
            choice = m
    return N.MSP_EIGH_JACOBI if choice == "jacobi" else N.MSP_EIGH_DC


def main(argv=None):
    ap = argparse.ArgumentParser(description=__doc__.splitlines()[0])
    ap.add_argument("--out", default=DEFAULT_PATH)
    ap.add_argument("--quick", action="store_true", help="fewer batch sizes, no chunk sweep")
    args = ap.parse_args(argv)
    res = tune(quick=args.quick)
    with open(args.out, "w") as f:
        json.dump(res, f, indent=1, sort_keys=True)
    print(json.dumps({k: v for k, v in res.items() if k != "measured"}), flush=True)


if __name__ == "__main__":
    main()
