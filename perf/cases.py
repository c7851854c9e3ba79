"""Performance cases of the library: the calls that programs make of it, over
the range of sizes, bucket counts, element widths and key distributions that
the tests and bench.py use.

``listed()`` names the fixed cases and ``draw(rng)`` gives another one of the
same ranges.  A case is a dict of plain values:

* ``op``: multisplit, sort, compaction, histogram_bins, histogram_even,
  histogram_range or batch;
* ``n``: elements (the largest instance for a batch);
* ``key_bytes`` / ``value_bytes``: 4 or 8; 0 value bytes means key-only;
* ``buckets``, ``identifier`` (range, delta or digit) and ``keys`` (uniform,
  zipf over the buckets, or sorted);
* ``offsets``: the bucket starts go to the host (a blocking call, as the
  reference's API), to the device, or nowhere;
* ``shift``: the inputs start this many elements into their allocation, as a
  slice of a larger array does.

All outputs are whole numbers: permuted keys and values, counts, starts.
"""
import math

import numpy as np
import torch

import gpumultisplit_amd as gms


def listed():
    return [
        # The smallest call: a few hundred to a few thousand items sorted into
        # a handful of bins inside a larger GPU program, starts kept on the
        # device.  Nothing but launches and latency.
        dict(name="multisplit_ko_8_1k", op="multisplit", n=1021, key_bytes=4, value_bytes=0,
             buckets=8, identifier="range", keys="uniform", offsets="device", shift=0),
        # The reference's call form at a medium size: key-value, bucket starts
        # handed to the host, which waits for them (a frontier or tile binning
        # step whose next launches depend on the counts).
        dict(name="multisplit_kv_64_60k", op="multisplit", n=60013, key_bytes=4, value_bytes=4,
             buckets=64, identifier="delta", keys="uniform", offsets="host", shift=0),
        # A partitioning step on a million skewed rows (a hash-join or a
        # shuffle partition with popular keys).
        dict(name="multisplit_kv_256_1m_zipf", op="multisplit", n=1 << 20, key_bytes=4,
             value_bytes=4, buckets=256, identifier="range", keys="zipf", offsets="device",
             shift=0),
        # The largest partitioning step, the benchmark's default workload.
        dict(name="multisplit_kv_256_128m", op="multisplit", n=1 << 27, key_bytes=4,
             value_bytes=4, buckets=256, identifier="range", keys="uniform", offsets="none",
             shift=0),
        # More buckets than one pass takes: grid cells or graph vertices as
        # buckets, a few million elements.
        dict(name="multisplit_kv_4096_3m", op="multisplit", n=3000017, key_bytes=4,
             value_bytes=4, buckets=4096, identifier="range", keys="uniform", offsets="device",
             shift=0),
        # Rows with 64-bit keys and 64-bit payloads.
        dict(name="multisplit_kv64_256_16m", op="multisplit", n=(1 << 24) + 5, key_bytes=8,
             value_bytes=8, buckets=256, identifier="range", keys="uniform", offsets="device",
             shift=0),
        # A small radix sort, the common size of a per-block or per-request sort.
        dict(name="sort8_ko_5k", op="sort", n=5003, key_bytes=4, value_bytes=0, digit_bits=8,
             keys="uniform", shift=0),
        # 64-bit keys with 32-bit indices, the argsort of a few hundred
        # thousand ids or timestamps.
        dict(name="sort8_k64v32_300k", op="sort", n=300007, key_bytes=8, value_bytes=4,
             digit_bits=8, keys="uniform", shift=0),
        # The benchmark's radix sort.
        dict(name="sort8_kv_32m", op="sort", n=1 << 25, key_bytes=4, value_bytes=4, digit_bits=8,
             keys="uniform", shift=0),
        # Stream compaction that returns the kept count to the host.
        dict(name="compaction_ko_4m", op="compaction", n=(1 << 22) - 77, key_bytes=4,
             value_bytes=0, keep=0.5, keys="uniform", shift=0),
        # Custom-edge histogram of float samples, the reference's range driver.
        dict(name="histogram_range_64m", op="histogram_range", n=(1 << 26) + 1, bins=256, shift=0),
        # A batch of uneven multisplits and sorts (one per query, image or
        # expert), planned once and run again on new contents.
        dict(name="batch_256_mixed", op="batch", count=256, sorts=64, n=1 << 18, buckets=64,
             value_bytes=4, keys="uniform"),
    ]


def _log_int(rng, lo, hi):
    """A whole number in [lo, hi], spread evenly over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["multisplit"] * 5 + ["sort"] * 3 +
                    ["compaction", "histogram_bins", "histogram_even", "histogram_range", "batch"])
    shift = rng.choice([0, 0, 0, 0, 1, 3])
    keys = rng.choice(["uniform", "uniform", "uniform", "zipf", "sorted"])
    if op == "multisplit":
        kb, vb = rng.choice([(4, 4), (4, 4), (4, 0), (4, 0), (8, 8), (8, 0), (8, 4), (4, 8)])
        buckets = rng.choice([2, 3, 8, 10, 16, 32, 33, 64, 100, 128, 200, 256, 256, 512, 1000,
                              1024, 2048, 5000, 1 << 16, 1 << 18, 1 << 20])
        # the passes of many buckets and the width of an element bound the size
        cost = max(1, -(-(buckets - 1).bit_length() // 8)) * (kb + vb) / 8
        return dict(op=op, n=_log_int(rng, 256, int((1 << 27) / cost)), key_bytes=kb,
                    value_bytes=vb, buckets=buckets,
                    identifier=rng.choice(["range", "range", "delta"]), keys=keys,
                    offsets=rng.choice(["host", "device", "none"]), shift=shift)
    if op == "sort":
        kb, vb = rng.choice([(4, 4), (4, 4), (4, 0), (4, 0), (8, 8), (8, 0), (8, 4)])
        bits = rng.choice([8, 8, 8, 7, 6])
        cost = (kb * 8 / 32) * (8 / bits) * (kb + vb) / 8
        return dict(op=op, n=_log_int(rng, 256, int((1 << 25) / cost)), key_bytes=kb,
                    value_bytes=vb, digit_bits=bits, keys="sorted" if keys == "sorted" else "uniform",
                    shift=shift)
    if op == "compaction":
        return dict(op=op, n=_log_int(rng, 256, 1 << 27), key_bytes=4, value_bytes=rng.choice([0, 4]),
                    keep=rng.choice([0.05, 0.3, 0.5, 0.95]), keys="uniform", shift=shift)
    if op == "batch":
        top = rng.choice([1 << 12, 1 << 16, 1 << 18, 1 << 20])
        count = _log_int(rng, 16, 512)
        return dict(op=op, count=count, sorts=rng.choice([0, 0, count // 4]), n=top,
                    buckets=rng.choice([2, 16, 64, 256]), value_bytes=rng.choice([0, 4, 4]),
                    keys="uniform")
    return dict(op=op, n=_log_int(rng, 256, 1 << 27), bins=rng.choice([10, 64, 200, 256]), shift=shift)


# ------------------------------------------------------------------- inputs
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _words(n, elem_bytes, g):
    """n uniform elements over the whole range of their width."""
    if elem_bytes == 4:
        return torch.randint(-(1 << 31), 1 << 31, (n,), dtype=torch.int32, device="cuda", generator=g)
    return torch.randint(-(1 << 63), (1 << 63) - 1, (n,), dtype=torch.int64, device="cuda", generator=g)


def _keys(case, n, g):
    kb, kind = case["key_bytes"], case["keys"]
    if kind == "zipf":
        # a Zipf(1.1) bucket per key, then a key inside that bucket's range
        B = case["buckets"]
        w = 1.0 / torch.arange(1, B + 1, dtype=torch.float64, device="cuda") ** 1.1
        cdf = (torch.cumsum(w, 0) / w.sum()).to(torch.float32)
        u = torch.rand(n, device="cuda", generator=g)
        b = torch.searchsorted(cdf, u).clamp_(max=B - 1)
        width = (1 << 32) // B
        k = b * width + torch.randint(0, width, (n,), dtype=torch.int64, device="cuda", generator=g)
        if kb == 8:
            return k * (1 << 32) + torch.randint(0, 1 << 32, (n,), dtype=torch.int64, device="cuda",
                                                 generator=g)
        return k.to(torch.int32)
    k = _words(n, kb, g)
    if kind == "sorted":
        # ascending as unsigned numbers
        lowest = -(1 << (8 * kb - 1))
        k = torch.sort(k).values ^ lowest
    return k


def _identifier(case):
    B, bits = case["buckets"], 8 * case["key_bytes"]
    if case["identifier"] == "delta":
        return gms.delta_func(max(1, -(-(1 << bits) // B)))
    return gms.range_bucket(B)


def _slice(t, shift):
    """The same contents, `shift` elements into an allocation."""
    if not shift:
        return t
    big = torch.empty(t.numel() + shift, dtype=t.dtype, device=t.device)
    big[shift:] = t
    return big[shift:]


def _values(n, elem_bytes):
    return torch.arange(n, dtype=torch.int32 if elem_bytes == 4 else torch.int64, device="cuda")


def _batch_sizes(case):
    """Uneven sizes 2^U, U uniform in [8, log2 n]: the same ones for every seed."""
    r = np.random.Generator(np.random.PCG64(case["count"]))
    return np.rint(2.0 ** r.uniform(8.0, math.log2(case["n"]), case["count"])).astype(int)


def prepare(case, seed):
    op, g, s = case["op"], _generator(seed), {"case": case}
    if op == "batch":
        sizes = _batch_sizes(case)
        starts = np.concatenate([[0], np.cumsum((sizes + 3) // 4 * 4)])  # 16-byte boundaries
        span, vb = int(starts[-1]), case["value_bytes"]
        s["kin"] = _words(span, 4, g)
        s["kout"] = torch.zeros_like(s["kin"])
        s["vin"] = _values(span, 4) if vb else None
        s["vout"] = torch.zeros_like(s["vin"]) if vb else None
        f = gms.range_bucket(case["buckets"])
        items, sorts = [], []
        for i, (a, n) in enumerate(zip(starts[:-1].tolist(), sizes.tolist())):
            ki, ko = s["kin"][a:a + n], s["kout"][a:a + n]
            v = dict(d_value_in=s["vin"][a:a + n], d_value_out=s["vout"][a:a + n]) if vb else {}
            if i < case["sorts"]:
                sorts.append(gms.BatchSortItem(ki, ko, n, 8, **v))
            else:
                items.append(gms.BatchItem(ki, ko, n, case["buckets"], f, **v))
        s["batch"] = gms.Batch(items, sorts=sorts)
        return s
    n, shift = case["n"], case["shift"]
    if op.startswith("histogram"):
        bins = case["bins"]
        s["hist"] = torch.zeros(bins, dtype=torch.int32, device="cuda")
        if op == "histogram_bins":
            s["x"] = _slice(_words(n, 4, g), shift)
            s["f"] = gms.range_bucket(bins)
            return s
        s["x"] = _slice(torch.rand(n, device="cuda", generator=g) * 1024.0, shift)
        if op == "histogram_range":
            lv = torch.sort(torch.rand(bins + 1, device="cuda", generator=g) * 1024.0).values
            lv[0], lv[-1] = 0.0, 1024.0
            s["levels"] = lv
        return s
    kb, vb = case["key_bytes"], case["value_bytes"]
    s["kin"] = _slice(_keys(case, n, g), shift)
    s["kout"] = torch.empty_like(s["kin"])
    s["vin"] = _slice(_values(n, vb), shift) if vb else None
    s["vout"] = torch.empty_like(s["vin"]) if vb else None
    if op == "multisplit":
        s["f"] = _identifier(case)
        s["ctx"] = gms.multisplit_context(case["buckets"])
        (gms.multisplit_allocate_key_value if vb else gms.multisplit_allocate_key_only)(n, s["ctx"])
        if case["offsets"] == "host":
            s["starts"] = np.zeros(case["buckets"], dtype=np.uint32)
        elif case["offsets"] == "device":
            s["starts"] = torch.empty(case["buckets"], dtype=torch.int32, device="cuda")
    elif op == "sort":
        api = "multisplit_sort_%dbit" % case["digit_bits"]
        s["ctx"] = gms.ms_sort_context()
        if vb:
            getattr(gms, api + "_allocate_pairs")(n, s["ctx"], key_bytes=kb, value_bytes=vb)
            s["sort"] = getattr(gms, api + "_pairs")
        else:
            getattr(gms, api + "_allocate")(n, s["ctx"], key_bytes=kb)
            s["sort"] = getattr(gms, api)
    else:
        s["f"] = gms.delta_func(int(case["keep"] * (1 << 32)))
        s["ctx"] = gms.compaction_context()
        (gms.compaction_allocate_key_value if vb else gms.compaction_allocate_key_only)(n, s["ctx"])
    return s


# --------------------------------------------------------------------- pass
def run(s):
    case = s["case"]
    op = case["op"]
    if op == "batch":
        s["batch"].run()
        return [s["kout"]] if s["vout"] is None else [s["kout"], s["vout"]]
    n = case["n"]
    if op.startswith("histogram"):
        s["hist"].zero_()  # the histograms add to what is there
        if op == "histogram_bins":
            gms.histogram(s["x"], n, s["hist"], case["bins"], s["f"])
        elif op == "histogram_even":
            gms.multisplit2_histogram_even(s["x"], n, s["hist"], 0.0, 1024.0, case["bins"] / 1024.0,
                                           case["bins"])
        else:
            gms.multisplit2_histogram_range(s["x"], n, s["hist"], s["levels"], case["bins"] + 1)
        return s["hist"]
    kin, kout, vin, vout, ctx = s["kin"], s["kout"], s["vin"], s["vout"], s["ctx"]
    if op == "multisplit":
        if case["offsets"] == "host":
            if vin is None:
                gms.multisplit_key_only(kin, kout, n, ctx, s["f"], s["starts"])
            else:
                gms.multisplit_key_value(kin, vin, kout, vout, n, ctx, s["f"], s["starts"])
        elif case["offsets"] == "device":
            gms.multisplit(kin, kout, n, ctx, s["f"], vin, vout, s["starts"])
        elif vin is None:
            gms.multisplit_key_only(kin, kout, n, ctx, s["f"])
        else:
            gms.multisplit_key_value(kin, vin, kout, vout, n, ctx, s["f"])
        out = [kout] if vout is None else [kout, vout]
        return out + [s["starts"]] if "starts" in s else out
    if op == "sort":
        if vin is None:
            s["sort"](kin, kout, n, ctx)
            return [kout]
        s["sort"](kin, kout, vin, vout, n, ctx)
        return [kout, vout]
    if vin is None:
        return [gms.compaction_key_only(kin, kout, n, ctx, s["f"]), kout]
    return [gms.compaction_key_value(kin, vin, kout, vout, n, ctx, s["f"]), kout, vout]


def work(case):
    """Each input element read once and each output element written once."""
    op = case["op"]
    if op == "batch":
        return {"bytes": 2 * int(_batch_sizes(case).sum()) * (4 + case["value_bytes"]), "flops": 0}
    if op.startswith("histogram"):
        return {"bytes": 4 * case["n"] + 8 * case["bins"], "flops": 0}
    b = 2 * case["n"] * (case["key_bytes"] + case["value_bytes"])
    if op == "multisplit" and case["offsets"] != "none":
        b += 4 * case["buckets"]
    return {"bytes": b, "flops": 0}
