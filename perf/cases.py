"""Performance cases of the VBSR SpMM library: C = A*B through its public entry points.

A case names a matrix family (block rows and columns, blocks per block row, block sizes, column pattern), the RHS width
and the entry point.  The families are those of the library's own generator, and "skewed" matrices, whose block rows
hold very different numbers of blocks (none in some).  A program builds the device matrix and the plan once and then
multiplies panel after panel, so both belong to `prepare` and a pass is one product.
"""

import math

import numpy as np
import torch

import varblockspmm_amd as vb

RHS = (8, 16, 32, 64)
DEGREES = (1, 2, 4, 8, 16)
MEAN_SIZE = {"uniform": 32.0, "low": 32.0, "high": 36.0, "tied8to64": 36.0, "bimodal": 34.0, "bimodal8or64": 36.0}
EXTENTS = {"uniform": (32,), "low": (24, 32, 40), "high": tuple(range(8, 65, 8)), "tied8to64": tuple(range(8, 65, 8)),
           "bimodal": (8, 16, 48, 64), "bimodal8or64": (8, 64)}
SKEW = 1.25  # of the logarithm of the row lengths
# The most blocks * RHS of one case, which bounds a drawn case's cost by the largest listed one's.
MOST_BLOCK_COLUMNS = 8192 * 16 * 64


def listed():
    def case(name, rows, degree, sizes, pattern, rhs, call="plan", cols=None):
        return {"name": name, "rows": rows, "cols": cols or rows, "degree": degree, "sizes": sizes, "pattern": pattern,
                "rhs": rhs, "call": call}

    return [
        # The smallest products: a test-sized matrix, where a pass is its launch.
        case("smallest", 48, 4, "high", "local", 8),
        # A small band matrix, one panel of eight vectors: the size a host can still do by itself.
        case("band_1024_rhs8", 1024, 4, "high", "clamped", 8),
        # A medium matrix with near-uniform blocks.
        case("medium_1024_rhs16", 1024, 8, "low", "random", 16),
        # Few, long block rows (a coarse level, or one device's share of a matrix) and an odd number of them.
        case("few_rows_203_rhs32", 203, 16, "high", "random", 32),
        # The same kind of matrix through the kernel a caller selects for it: split rows and a workspace.
        case("split_row_64_rhs64", 64, 16, "high", "random", 64, "split_row"),
        # The width where A is nearly all of the traffic, at full size.
        case("full_4096_rhs8", 4096, 8, "high", "random", 8),
        # The library's headline product.
        case("full_4096_rhs32", 4096, 8, "high", "random", 32),
        # One block a row: a block-diagonal or permutation-like operator.
        case("degree1_4096_rhs16", 4096, 1, "tied8to64", "random", 16),
        # Wide panel, many blocks a row, the smallest and largest blocks mixed.
        case("wide_4096_rhs64", 4096, 16, "bimodal8or64", "random", 64),
        # Rows of very different lengths and a rectangular matrix of odd extents.
        case("skewed_3001_rhs16", 3001, 8, "high", "skewed", 16, cols=2503),
        # The order-preserving kernel, for callers who need the sums in the reference's order bit for bit.
        case("ordered_4096_rhs32", 4096, 8, "high", "random", 32, "ordered"),
        # The largest: a wide band matrix with wide panels.
        case("largest_8192_rhs64", 8192, 16, "low", "clamped", 64),
    ]


def draw(rng):
    while True:
        rows = int(round(math.exp(rng.uniform(math.log(32), math.log(8192)))))
        cols = rows if rng.random() < 0.7 else max(32, int(rows * math.exp(rng.uniform(-0.7, 0.7))))
        degree = rng.choice(DEGREES)
        rhs = rng.choice(RHS)
        pattern = rng.choice(("random", "random", "local", "clamped", "skewed"))
        sizes = rng.choice(tuple(MEAN_SIZE))
        call = rng.choice(("plan",) * 6 + ("ordered", "split_row"))
        if call == "split_row" and (rows > 256 or degree < 8):
            continue  # callers split few, long rows
        if pattern in ("local", "clamped") and cols <= 2 * degree:
            continue
        if rows * degree * rhs <= MOST_BLOCK_COLUMNS // (4 if call == "ordered" else 1):
            return {"rows": rows, "cols": cols, "degree": degree, "sizes": sizes, "pattern": pattern, "rhs": rhs,
                    "call": call}


def _columns(rng, case, degree):
    """Each block row's distinct block columns, ascending, row after row."""
    rows, cols = case["rows"], case["cols"]
    if case["pattern"] in ("random", "skewed"):
        return np.concatenate([np.sort(rng.choice(cols, d, replace=False)) for d in degree])
    # A window of `degree` columns to either side of the diagonal: cyclic ("local") or clamped at the edges.
    d = case["degree"]
    offsets = np.argsort(rng.random((rows, 2 * d + 1)), axis=1)[:, :d]
    diagonal = np.arange(rows)[:, None]
    if case["pattern"] == "local":
        picked = (diagonal + offsets - d) % cols
    else:
        picked = np.clip(diagonal, d, cols - 1 - d) + offsets - d
    return np.sort(picked, axis=1).reshape(-1)


def _host(case, seed):
    """The matrix, as a program that assembled it would hold it: values uniform in [-1, 1].

    The block sizes are the case's own, so that every seed's panels have the same shape; which blocks a row holds, how
    many it holds where rows are skewed, and the values come from the seed."""
    rows, cols = case["rows"], case["cols"]
    extents = np.array(EXTENTS[case["sizes"]])
    rng = np.random.default_rng([rows, cols, case["degree"], case["rhs"]])
    row_size, col_size = rng.choice(extents, rows), rng.choice(extents, cols)
    rng = np.random.default_rng(seed)
    if case["sizes"] == "tied8to64":
        col_size[:min(rows, cols)] = row_size[:min(rows, cols)]
    if case["pattern"] == "skewed":
        # A long tail of row lengths, `degree` on average, from empty rows to some that hold tens of times that.
        raw = case["degree"] * rng.lognormal(-0.5 * SKEW * SKEW, SKEW, rows) + rng.random(rows)
        degree = np.minimum(raw, cols // 2).astype(np.int64)
    else:
        degree = np.full(rows, case["degree"])
    row_ptr = np.concatenate([[0], np.cumsum(degree)])
    block_col = _columns(rng, case, degree)
    owner = np.repeat(np.arange(rows), degree)
    value_off = np.concatenate([[0], np.cumsum(row_size[owner] * col_size[block_col])])
    values = rng.random(int(value_off[-1]), dtype=np.float32)
    values *= 2
    values -= 1
    return vb.HostMatrix(rows, cols, row_ptr=row_ptr, block_col=block_col, row_size=row_size, col_size=col_size,
                         row_scalar_off=np.concatenate([[0], np.cumsum(row_size)]),
                         col_scalar_off=np.concatenate([[0], np.cumsum(col_size)]), value_off=value_off, values=values)


def _panel(host, case, seed, device):
    count = host.scalar_cols * case["rhs"]
    return torch.from_numpy(np.random.default_rng([seed, 1]).random(count, dtype=np.float32) * 2 - 1).to(device)


def prepare(case, seed):
    host = _host(case, seed)
    state = {"call": case["call"], "rhs": case["rhs"], "matrix": vb.Matrix(host), "B": _panel(host, case, seed, "cuda"),
             "C": torch.empty(host.scalar_rows * case["rhs"], dtype=torch.float32, device="cuda")}
    if case["call"] == "ordered":
        state["view"] = state["matrix"].device_view()
    else:
        state["plan"] = vb.Plan(state["matrix"], case["rhs"],
                                kernel="split_row" if case["call"] == "split_row" else "auto")
    return state


def run(state):
    if state["call"] == "ordered":
        vb.launch_row_owned_scalar(state["view"], state["B"], state["C"], state["rhs"])
    else:
        state["plan"].execute(state["B"], state["C"])
    return state["C"]


def work(case):
    """Expected bytes (A, B and C once, the format's own arrays) and flops over the case's random sizes."""
    size, rows, cols, rhs = MEAN_SIZE[case["sizes"]], case["rows"], case["cols"], case["rhs"]
    blocks = rows * case["degree"]
    # Tied sizes share a row's and a column's draw, which matters only on the diagonal: the means still multiply.
    values = blocks * size * size
    arrays = 12 * (rows + 1) + 12 * (cols + 1) + 4 * rows + 12 * blocks
    return {"bytes": 4.0 * (values + rhs * size * (rows + cols)) + arrays, "flops": 2.0 * rhs * values}


def tolerance(case):
    # The order-preserving kernel promises one order of sums; the others may sum in any order, in FP32 throughout.
    return "exact" if case["call"] == "ordered" else {"rel": 2e-6, "max": 4e-5}


def exact(case, seed):
    device = "cuda" if torch.cuda.is_available() else "cpu"
    host = _host(case, seed)
    rhs, m = case["rhs"], host.scalar_rows
    b = _panel(host, case, seed, device).double().view(rhs, host.scalar_cols)
    values = torch.from_numpy(host.values).to(device)
    out = torch.zeros(rhs, m, dtype=torch.float64, device=device)
    owner = np.repeat(np.arange(host.block_rows), np.diff(host.row_ptr))
    heights, widths = host.row_size[owner], host.col_size[host.block_col]
    for h in np.unique(heights):
        for w in np.unique(widths):
            which = np.nonzero((heights == h) & (widths == w))[0]
            for part in np.array_split(which, max(1, len(which) // 4096)):
                if not len(part):
                    continue
                index = lambda starts, n: (torch.from_numpy(starts.astype(np.int64)).to(device)[:, None] +  # noqa: E731
                                           torch.arange(int(n), device=device)[None, :])
                a = values[index(host.value_off[part], h * w)].double().view(len(part), int(w), int(h))
                k = index(host.col_scalar_off[host.block_col[part]], w).reshape(-1)
                panel = b[:, k].view(rhs, len(part), int(w)).transpose(0, 1).contiguous()
                rows = index(host.row_scalar_off[owner[part]], h).reshape(-1)
                out.index_add_(1, rows, torch.bmm(panel, a).transpose(0, 1).reshape(rhs, -1))
    return out.reshape(-1)
