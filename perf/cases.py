"""Performance cases of the kernel library: calls that programs on top of it make.

listed() gives fixed cases, draw(rng) further ones of the same ranges,
prepare(case, seed) the matrix, block vectors and handles a program holds
before the call, run(state) one pass through the public entry points,
work(case) the bytes and flops of a pass, and exact(case, seed) the result in
64 bits with plain torch.

Every case is a kind of call ("op"):

  spmv     y = alpha A x + beta y                      sparseMat_times_mvec
  shift    y = alpha (A + diag(s)) x + beta y          sparseMat_times_mvec_vadd_mvec
  dots     y = alpha A x + beta y, <y,y>, <x,y>        fused_spmv_mvdot
  update   Y(:,c) += a_c X(:,c), then ||Y(:,c)||       mvec_vadd_mvec, mvec_norm2
  mix      W = V C                                     mvec_times_sdMat
  cgs      twice: C = V'W, W -= V C                    mvecT_times_mvec, mvec_times_sdMat
  cholqr   V = Q R                                     chol_QR
  carp     forward + backward Kaczmarz sweep           carp_sweep
  minres   (A + s_j I) x_j = b_j, iteration limit      blockedMINRES_shifted
  gmres    (A + s_j I) x_j = b_j, one restart cycle    blockedGMRES_shifted
  jada     smallest eigenvalues to 1e-8                subspacejada
"""
import ctypes
import math

import numpy as np
import torch

import phist_amd

DEV = "cuda"
ON_DEVICE = phist_amd.MVEC_RUN_ON_DEVICE


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------
def lap(nx, ny, nz):
    return {"matrix": "lap", "nx": nx, "ny": ny, "nz": nz}


def banded(n, nnz, halfband):
    return {"matrix": "banded", "n": n, "nnz": nnz, "halfband": halfband}


def spin(length, nup):
    return {"matrix": "spin", "length": length, "nup": nup}


def honey(w, length, long_range=0):
    return {"matrix": "honey", "w": w, "length": length, "long_range": long_range}


def listed():
    return [
        # a step of a small iterative solve, a coarse grid: launches and the wait for the dots count
        {"name": "dots_lap32_k4", "op": "dots", "dtype": "f64", "k": 4, "alpha": 1.0, "beta": 0.0, **lap(32, 32, 32)},
        # the kernel benchmark of the library: wide band, block of 8, both dots back on the host
        {"name": "dots_band4m_k8", "op": "dots", "dtype": "f64", "k": 8, "alpha": 1.0, "beta": 0.0,
         **banded(4194304, 32, 50000)},
        # operator of an FP32 correction equation on the 24-spin chain, one shift per column
        {"name": "shift_spin24_k4_f32", "op": "shift", "dtype": "f32", "k": 4, "alpha": 1.0, "beta": 0.0,
         **spin(24, 12)},
        # residuals of five systems on an odd-sized sheet: odd width, y read and written
        {"name": "spmv_sheet_k5", "op": "spmv", "dtype": "f64", "k": 5, "alpha": -1.0, "beta": 1.0,
         **honey(1499, 1001)},
        # vector update and norms of a block of four (the 24-spin chain's length)
        {"name": "update_2m7_k4", "op": "update", "dtype": "f64", "n": 2704156, "k": 4},
        # Cholesky QR of a tall block
        {"name": "cholqr_16m_k8", "op": "cholqr", "dtype": "f64", "n": 16777216, "k": 8},
        # thick restart of an eigensolver: 48 basis vectors to 24
        {"name": "restart_2m7_48to24", "op": "mix", "dtype": "f64", "n": 2704156, "k": 48, "m": 24},
        # four new directions against forty basis vectors, classical Gram-Schmidt twice
        {"name": "cgs_2m7_40p4", "op": "cgs", "dtype": "f64", "n": 2704156, "k": 40, "m": 4},
        # Kaczmarz sweep on a graphene sheet with long-range hopping
        {"name": "carp_graphene1024_k8", "op": "carp", "dtype": "f64", "k": 8, **honey(1024, 1024, 1)},
        # 32 shifted systems on an 8-million-site sheet, the largest block
        {"name": "minres_sheet8m_k32", "op": "minres", "dtype": "f64", "k": 32, "iters": 8, **honey(2000, 4000)},
        # one GMRES(30) cycle on 16 shifted systems of the 128^3 Laplacian
        {"name": "gmres_lap128_k16", "op": "gmres", "dtype": "f64", "k": 16, "iters": 30, **lap(128, 128, 128)},
        # eight smallest eigenvalues of a box, the whole eigensolver
        {"name": "jada_box64", "op": "jada", "dtype": "f64", "inner_f32": False, "eigs": 8, **lap(64, 58, 51)},
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def matrix():
        kind = rng.choice(("lap", "banded", "spin", "honey"))
        if kind == "lap":
            return lap(size(8, 160), size(8, 160), size(8, 160))
        if kind == "banded":
            n = size(4000, 3000000)
            return banded(n, rng.randint(5, 32), min(size(40, 50000), n // 4))
        if kind == "spin":
            length = rng.randint(12, 24)
            return spin(length, length // 2 - rng.randint(0, 2))
        return honey(size(48, 2000), size(48, 2000), rng.randint(0, 1))

    op = rng.choice(("spmv", "shift", "dots", "update", "mix", "cgs", "cholqr", "carp", "minres", "gmres", "jada"))
    dtype = rng.choice(("f64", "f64", "f32"))
    if op in ("spmv", "shift", "dots"):
        beta = rng.choice((0.0, 0.0, 1.0, 0.5))
        return {"op": op, "dtype": dtype, "k": rng.choice((1, 2, 3, 4, 4, 5, 6, 7, 8, 8, 12, 16, 32)),
                "alpha": rng.choice((1.0, -1.0)), "beta": beta, **matrix()}
    if op == "update":
        return {"op": op, "dtype": dtype, "n": size(3000, 8000000), "k": rng.choice((1, 2, 3, 4, 5, 8, 16, 32))}
    if op == "mix":
        k = rng.randint(1, 48)
        return {"op": op, "dtype": dtype, "n": size(3000, 4000000), "k": k, "m": rng.randint(1, k)}
    if op == "cgs":
        return {"op": op, "dtype": dtype, "n": size(5000, 2700000), "k": rng.randint(2, 44), "m": rng.randint(1, 8)}
    if op == "cholqr":
        return {"op": op, "dtype": dtype, "n": size(5000, 4000000), "k": rng.randint(1, 32)}
    if op == "carp":
        return {"op": op, "dtype": dtype, "k": rng.choice((1, 2, 3, 4, 8, 16)),
                **honey(size(48, 1024), size(48, 1024), rng.randint(0, 1))}
    if op == "minres":
        return {"op": op, "dtype": "f64", "k": rng.randint(1, 32), "iters": rng.randint(4, 12),
                **honey(size(64, 2000), size(64, 2000))}
    if op == "gmres":
        return {"op": op, "dtype": "f64", "k": rng.randint(1, 16), "iters": rng.randint(8, 30),
                **lap(size(24, 110), size(24, 110), size(24, 110))}
    nz = rng.randint(20, 52)
    return {"op": "jada", "dtype": "f64", "inner_f32": rng.random() < 0.5, "eigs": 8,
            **lap(round(1.26 * nz), round(1.14 * nz), nz)}


# ---------------------------------------------------------------------------
# matrices: sizes, the library's generators, and the same entries with torch
# ---------------------------------------------------------------------------
def _rows(case):
    kind = case.get("matrix")
    if kind == "lap":
        return case["nx"] * case["ny"] * case["nz"]
    if kind == "spin":
        return math.comb(case["length"], case["nup"])
    if kind == "honey":
        return case["w"] * case["length"]
    return case["n"]


def _entries(case):
    """number of stored entries (exact for the Laplacian and the band, an upper bound at the edges otherwise)"""
    n = _rows(case)
    kind = case["matrix"]
    if kind == "lap":
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        return 7 * n - 2 * (nx * ny + ny * nz + nx * nz)
    if kind == "banded":
        return n * case["nnz"]
    if kind == "spin":
        length, up = case["length"], case["nup"]
        return n + 2 * length * math.comb(length - 2, up - 1)
    return n * (13 if case["long_range"] else 4)


def _matrix(be, case, seed):
    kind = case["matrix"]
    if kind == "lap":
        return be.laplace3d(case["nx"], case["ny"], case["nz"])
    if kind == "banded":
        return be.banded_random(case["n"], case["nnz"], case["halfband"], 40.0, seed)
    if kind == "spin":
        return be.spinchain_sz(case["length"], case["nup"])
    return be.honeycomb(case["w"], case["length"], 0, 0, case["long_range"], 1.0, seed)


_GOLDEN, _MIX1, _MIX2, _ROW = (int(np.uint64(v).astype(np.int64)) for v in (
    0x9E3779B97F4A7C15, 0xBF58476D1CE4E5B9, 0x94D049BB133111EB, 0xD1B54A32D192ED03))


def _shr(z, s):
    return (z >> s) & ((1 << (64 - s)) - 1)


def _splitmix(state):
    """next state and output of SplitMix64 (Steele, Lea & Flood), 64-bit words held in int64"""
    state = state + _GOLDEN
    z = (state ^ _shr(state, 30)) * _MIX1
    z = (z ^ _shr(z, 27)) * _MIX2
    return state, z ^ _shr(z, 31)


def _ell(case, seed, single):
    """the matrix as (col, val), each rows x width, padded with zeros at the row's own column"""
    n = _rows(case)
    i = torch.arange(n, device=DEV)
    kind = case["matrix"]
    cols, vals = [], []

    def add(ok, c, v):
        cols.append(torch.where(ok, c, i))
        vals.append(torch.where(ok, torch.as_tensor(v, dtype=torch.float64, device=DEV), 0.0))

    if kind == "lap":
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        x, y, z = i % nx, (i // nx) % ny, i // (nx * ny)
        add(i >= 0, i, 6.0)
        for p, top, step in ((x, nx, 1), (y, ny, nx), (z, nz, nx * ny)):
            add(p > 0, i - step, -1.0)
            add(p < top - 1, i + step, -1.0)
    elif kind == "spin":
        length, up = case["length"], case["nup"]
        words = torch.arange(1 << length, device=DEV, dtype=torch.int32)
        ones = torch.zeros_like(words)
        for b in range(length):
            ones += (words >> b) & 1
        words = words[ones == up].long()
        index = torch.zeros(1 << length, device=DEV, dtype=torch.int64)
        index[words] = i
        diag = torch.zeros(n, device=DEV, dtype=torch.float64)
        for b in range(length):
            bond = (1 << b) | (1 << ((b + 1) % length))
            anti = ((words >> b) & 1) != ((words >> ((b + 1) % length)) & 1)
            diag += torch.where(anti, -1.0, 1.0).double()
            add(anti, index[words ^ bond], 2.0)
        add(i >= 0, i, diag)
    elif kind == "honey":
        w_, l_ = case["w"], case["length"]
        far = case["long_range"] != 0
        t1, t2, t3 = -1.0, -0.1 / 2.78, -0.095 / 2.78
        row, col = i // w_, i % w_
        up = (row + col) % 2 != 0

        def hop(dl, dw, a, ok):
            r, c = row + dl, col + dw
            add(ok & (r >= 0) & (r < l_) & (c >= 0) & (c < w_), r * w_ + c, a)

        every = i >= 0
        for dl in (-1, 1):
            bonded = up if dl > 0 else ~up
            hop(dl, 0, t1, bonded)
            if far:
                hop(dl, 0, t3, ~bonded)
                hop(dl, -1, t2, every)
                hop(dl, 1, t2, every)
                hop(dl, -2, t3, bonded)
                hop(dl, 2, t3, bonded)
        for dw in (-1, 1):
            hop(0, dw, t1, every)
            if far:
                hop(0, 2 * dw, t2, every)
        _, z = _splitmix((i + 1) * _ROW ^ seed)
        u = _shr(z, 11).double() * 2.0 ** -53
        add(every, i, 1.0 * (u - 0.5) + (3.0 * t3 if far else 0.0))
    else:
        want, half = case["nnz"], case["halfband"]
        lo, hi = (i - half).clamp(min=0), (i + half).clamp(max=n - 1)
        width = hi - lo + 1
        c_all = i[:, None].repeat(1, want)
        v_all = torch.zeros(n, want, device=DEV, dtype=torch.float64)
        v_all[:, 0] = 40.0
        have = torch.ones_like(i)
        state = (i + 1) * _ROW ^ seed
        live = i
        while live.numel():
            wd = width[live]
            s, z = _splitmix(state[live])
            c = lo[live] + ((_shr(z, 32) % wd) * ((1 << 32) % wd) + (z & 0xFFFFFFFF) % wd) % wd
            fresh = (c_all[live] != c[:, None]).all(1)  # unused slots hold the row's own index
            at, k = live[fresh], have[live[fresh]]
            state[live] = s
            s, z = _splitmix(state[at])
            state[at] = s
            c_all[at, k] = c[fresh]
            v_all[at, k] = _shr(z, 11).double() * 2.0 ** -52 - 1.0
            have[at] += 1
            live = live[have[live] < want]
        return c_all, v_all.float().double() if single else v_all
    col, val = torch.stack(cols, 1), torch.stack(vals, 1)
    return col, val.float().double() if single else val


def _times(ell, x):
    col, val = ell
    y = torch.zeros_like(x)
    for j in range(col.shape[1]):
        y += val[:, j:j + 1] * x[col[:, j]]
    return y


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _uniform(seed, part, rows, cols, dtype):
    """rows x cols numbers of U(-1, 1) from the seed, another stream for each part"""
    g = torch.Generator(device=DEV)
    g.manual_seed((seed * 1000003 + part) % (1 << 62))
    return torch.rand(rows, cols, generator=g, device=DEV, dtype=dtype) * 2 - 1


def _dtype(case):
    return torch.float64 if case["dtype"] == "f64" else torch.float32


def _shifts(case, seed):
    k = case["k"]
    if case["op"] == "gmres":
        return np.linspace(0.05, 1.0, k)
    return np.random.RandomState(seed % (1 << 31)).uniform(-2.5, 2.5, k)


def _inputs(case, seed):
    """the block vectors and small matrices that go into the call, as torch tensors"""
    op, dt, n = case["op"], _dtype(case), _rows(case)
    if op in ("spmv", "shift", "dots"):
        return {"x": _uniform(seed, 1, n, case["k"], dt), "y": _uniform(seed, 2, n, case["k"], dt)}
    if op == "update":
        return {"x": _uniform(seed, 1, n, case["k"], dt), "y": _uniform(seed, 2, n, case["k"], dt)}
    if op == "mix":
        return {"v": _uniform(seed, 1, n, case["k"], dt), "c": _uniform(seed, 2, case["k"], case["m"], dt)}
    if op == "cgs":
        v = _uniform(seed, 1, n, case["k"], torch.float64)
        for _ in range(2):  # an orthonormal basis by Cholesky QR, twice
            r = torch.linalg.cholesky((v.T @ v).cpu())
            v = v @ torch.linalg.inv(r).T.contiguous().to(DEV)
        return {"v": v.to(dt), "w": _uniform(seed, 2, n, case["m"], dt)}
    if op == "cholqr":
        return {"v": _uniform(seed, 1, n, case["k"], dt)}
    if op == "carp":
        return {"x": _uniform(seed, 1, n, case["k"], dt), "b": _uniform(seed, 2, n, case["k"], dt)}
    if op == "jada":
        return {"v0": _uniform(seed, 1, n, 1, dt)}
    b = _uniform(seed, 1, n, case["k"], dt)
    return {"b": b / b.norm(dim=0)}


class Block:
    """a block vector of the library, and a torch tensor on the same memory"""

    def __init__(self, be, n, k):
        self.map = be.map(n)
        self.mvec = be.mvec(self.map, k)
        self.h = self.mvec.h
        raw, lda = ctypes.c_void_p(), ctypes.c_int32()
        be.call("mvec_extract_view", self.h, ctypes.byref(raw), ctypes.byref(lda), flags=ON_DEVICE)
        size = be.dtype.itemsize
        self.__cuda_array_interface__ = {"shape": (n, k), "strides": (lda.value * size, size), "version": 3,
                                         "typestr": "<f%d" % size, "data": (raw.value, False)}

    def tensor(self):
        return torch.as_tensor(self, device=DEV)  # the tensor keeps the block alive

    def __del__(self):
        self.mvec.delete()
        self.map.delete()


class State:
    """handles of one case; deleted with it"""

    def __init__(self, case, seed):
        self.case, self.op = case, case["op"]
        self.be = be = phist_amd.Backend(np.float64 if case["dtype"] == "f64" else np.float32)
        be.init()
        self.owned, self.block, self.out = [], {}, {}
        if "matrix" in case:
            self.A = self.own(_matrix(be, case, seed))
        for name, t in _inputs(case, seed).items():
            if name == "c":
                self.c = self.own(be.sdmat(*t.shape, data=t.cpu().numpy()))
            else:
                self.new(name, *t.shape).copy_(t)
        n = _rows(case)
        if self.op in ("shift", "minres", "gmres"):
            self.shifts = _shifts(case, seed)
        if self.op == "update":
            self.a = np.ascontiguousarray(np.linspace(-1.0, 1.0, case["k"] + 1)[:-1], be.dtype)
        elif self.op == "mix":
            self.new("w", n, case["m"])
        elif self.op == "cgs":
            self.new("q", n, case["m"])
            self.c = [self.own(be.sdmat(case["k"], case["m"])) for _ in range(2)]
        elif self.op == "cholqr":
            self.new("q", n, case["k"])
            self.r = self.own(be.sdmat(case["k"], case["k"]))
        elif self.op == "carp":
            self.sigma, self.omega = np.full(case["k"], 42.9), np.full(case["k"], 1.5)
            self.carp = self.own(be.carp_setup(self.A, self.sigma))
        elif self.op in ("minres", "gmres"):
            self.new("x", n, case["k"]).zero_()
        elif self.op == "jada" and case["inner_f32"]:  # the matrix's FP32 copy is made once
            b, x = Block(be, n, 1), Block(be, n, 1)
            torch.cuda.synchronize()
            be.minres_shifted(self.A, [0.0], b, x, 1.0, 1, fp32=True)
        torch.cuda.synchronize()

    def own(self, handle):
        self.owned.append(handle)
        return handle

    def new(self, name, n, k):
        self.block[name] = b = Block(self.be, n, k)
        self.out[name] = t = b.tensor()
        return t

    def __del__(self):
        for h in reversed(self.owned):
            h.delete()


def prepare(case, seed):
    return State(case, seed)


def run(s):
    be, op, case, b, out = s.be, s.op, s.case, s.block, s.out
    if op == "spmv":
        be.spmv(case["alpha"], s.A, b["x"], case["beta"], b["y"])
        return out["y"]
    if op == "shift":
        be.spmv_shifted(case["alpha"], s.A, s.shifts, b["x"], case["beta"], b["y"])
        return out["y"]
    if op == "dots":
        ww, vw = be.fused_spmv_mvdot(case["alpha"], s.A, b["x"].mvec, case["beta"], b["y"])
        return [out["y"], ww, vw]
    if op == "update":
        be.call("mvec_vadd_mvec", s.a.ctypes.data_as(ctypes.c_void_p), b["x"].h, be.s(1.0), b["y"].h)
        return [out["y"], be.norm2(b["y"].mvec)]
    if op == "mix":
        be.times_sdmat(1.0, b["v"], s.c, 0.0, b["w"])
        return out["w"]
    if op == "cgs":
        be.call("mvec_add_mvec", be.s(1.0), b["w"].h, be.s(0.0), b["q"].h)
        for c in s.c:
            be.gram(1.0, b["v"], b["q"], 0.0, c)
            be.times_sdmat(-1.0, b["v"], c, 1.0, b["q"])
        return [out["q"], s.c[0].get()]
    if op == "cholqr":
        be.call("mvec_add_mvec", be.s(1.0), b["v"].h, be.s(0.0), b["q"].h)
        be.call("chol_QR", b["q"].h, s.r.h)
        return [out["q"], s.r.get()]
    if op == "carp":
        s.carp.sweep(s.sigma, b["b"].mvec, b["x"].mvec, s.omega)
        return out["x"]
    if op == "minres":
        it, rr, _ = be.minres_shifted(s.A, s.shifts, b["b"], b["x"], 1e-14, case["iters"])
        return [out["x"], it, rr]
    if op == "gmres":
        b["x"].mvec.put_value(0.0)  # the initial guess
        it, rr, _ = be.gmres_shifted(s.A, s.shifts, b["b"], b["x"], 1e-14, case["iters"], restart=case["iters"])
        return [out["x"], it, rr]
    k = case["eigs"]
    ev, _, nconv, _, q, r = be.subspacejada(s.A, k, which="SR", tol=1e-8, block_size=4, min_bas=2 * k, max_bas=4 * k,
                                            max_iters=500, inner="GMRES", inner_max_iters=10,
                                            inner_fp32=case["inner_f32"], v0=b["v0"].mvec)
    q.delete()
    r.delete()
    return [np.sort(ev[:k]), nconv >= k]


# ---------------------------------------------------------------------------
# work and exact results
# ---------------------------------------------------------------------------
def work(case):
    """inputs once, outputs once; for the iterations of a solver the matrix and
    the blocks that each of their steps has to meet (a reduction over all rows
    lies between the product, the new basis vector and the solution)"""
    n, k, s, op = _rows(case), case.get("k", 1), 8 if case["dtype"] == "f64" else 4, case["op"]
    blk = n * k * s
    if "matrix" in case:
        nnz = _entries(case)
        mat = nnz * (s + 4) + 4 * n
    if op in ("spmv", "shift", "dots"):
        return {"bytes": mat + blk * (3 if case["beta"] else 2),
                "flops": 2 * nnz * k + (4 * n * k if op == "dots" else 0)}
    if op == "update":
        return {"bytes": 3 * blk, "flops": 4 * n * k}
    m = case.get("m", 0)
    if op == "mix":
        return {"bytes": n * s * (k + m), "flops": 2 * n * k * m}
    if op == "cgs":  # a reduction over all rows lies between the reads of the basis
        return {"bytes": n * s * (3 * k + 2 * m), "flops": 8 * n * k * m}
    if op == "cholqr":
        return {"bytes": 3 * blk, "flops": 4 * n * k * k}
    if op == "carp":
        return {"bytes": 2 * (mat + 3 * blk), "flops": 8 * nnz * k}
    it = case.get("iters", 1)
    if op == "minres":  # v -> w; w, v, v_old -> w; x, d -> x, d
        return {"bytes": it * (mat + 10 * blk), "flops": it * (2 * nnz * k + 16 * n * k)}
    if op == "gmres":  # v -> w; the basis twice (Gram-Schmidt twice)
        return {"bytes": it * (mat + 3 * blk) + it * (it + 1) * blk,
                "flops": it * 2 * nnz * k + 4 * it * (it + 1) * n * k}
    return {"bytes": mat + n * s * (1 + case["eigs"]), "flops": 2 * nnz * case["eigs"]}


def _pivoted_cholesky(g):
    """R with G = R'R, the largest remaining diagonal entry first (R(:, order) is upper triangular)"""
    g = g.copy()
    m = g.shape[0]
    r, left = np.zeros((m, m)), list(range(m))
    for row in range(m):
        p = max(left, key=lambda j: g[j, j])
        left.remove(p)
        r[row, p] = math.sqrt(g[p, p])
        for j in left:
            r[row, j] = g[p, j] / r[row, p]
        for j in left:
            g[left, j] -= r[row, left] * r[row, j]
    return r


def _exact_minres(ell, s, b, iters):
    """MINRES (Paige & Saunders) on every column"""
    beta1 = b.norm(dim=0)
    v, vold = b / beta1, torch.zeros_like(b)
    d1, d2, x = torch.zeros_like(b), torch.zeros_like(b), torch.zeros_like(b)
    beta = torch.zeros_like(beta1)
    c1, s1, c2, s2 = torch.ones_like(beta1), beta.clone(), torch.ones_like(beta1), beta.clone()
    phi = beta1.clone()
    for _ in range(iters):
        w = _times(ell, v) + v * s
        alpha = (w * v).sum(0)
        w = w - alpha * v - beta * vold
        bn = w.norm(dim=0)
        eps, dbar = s2 * beta, c2 * beta
        delta, gbar = c1 * dbar + s1 * alpha, c1 * alpha - s1 * dbar
        gamma = torch.hypot(gbar, bn)
        c2, s2, c1, s1 = c1, s1, gbar / gamma, bn / gamma
        d1, d2 = (v - delta * d1 - eps * d2) / gamma, d1
        x += c1 * phi * d1
        phi = -s1 * phi
        vold, v, beta = v, w / bn, bn
    return x, phi.abs() / beta1


def _exact_gmres(ell, s, b, m):
    """one cycle of GMRES(m) from x = 0 on every column"""
    k = b.shape[1]
    beta = b.norm(dim=0)
    basis, h = [b / beta], torch.zeros(k, m + 1, m, dtype=torch.float64)
    for i in range(m):
        w = _times(ell, basis[i]) + basis[i] * s
        for _ in range(2):
            c = [(v * w).sum(0) for v in basis]
            for v, a in zip(basis, c):
                w = w - a * v
            h[:, :i + 1, i] += torch.stack(c, 1).cpu()
        nrm = w.norm(dim=0)
        h[:, i + 1, i] = nrm.cpu()
        basis.append(w / nrm)
    rhs = torch.zeros(k, m + 1, 1, dtype=torch.float64)
    rhs[:, 0, 0] = beta.cpu()
    y = torch.stack([torch.linalg.lstsq(h[j], rhs[j], driver="gelsd").solution for j in range(k)])
    res = (rhs - torch.stack([h[j] @ y[j] for j in range(k)]))[:, :, 0].norm(dim=1)
    x = torch.zeros_like(b)
    for i in range(m):
        x += y[:, i, 0].to(DEV) * basis[i]
    return x, res / beta.cpu()


def exact(case, seed):
    op, n, single = case["op"], _rows(case), case["dtype"] == "f32"
    if op == "carp":  # the order of the rows is the library's own
        return None
    if op == "jada":
        one = [2 - 2 * np.cos(np.pi * np.arange(1, p + 1) / (p + 1)) for p in (case["nx"], case["ny"], case["nz"])]
        every = one[0][:9, None, None] + one[1][None, :9, None] + one[2][None, None, :9]
        return [np.sort(every.ravel())[:case["eigs"]], None]
    t = {name: v.double() for name, v in _inputs(case, seed).items()}
    if op == "update":
        a = np.linspace(-1.0, 1.0, case["k"] + 1)[:-1]
        a = torch.as_tensor(a.astype(np.float32 if single else np.float64), device=DEV).double()
        y = t["y"] + a * t["x"]
        return [y, y.norm(dim=0).cpu().numpy()]
    if op == "mix":
        return t["v"] @ t["c"]
    if op == "cgs":
        v, w = t["v"], t["w"]
        first = v.T @ w
        w = w - v @ first
        return [w - v @ (v.T @ w), first.cpu().numpy()]
    if op == "cholqr":
        v = t["v"]
        g = sum(p.T @ p for p in v.split(1 << 20)).cpu().numpy()
        r = _pivoted_cholesky(g)
        return [v @ torch.as_tensor(np.linalg.inv(r), device=DEV), r]
    ell = _ell(case, seed, single)
    if op in ("spmv", "shift", "dots"):
        y = _times(ell, t["x"])
        if op == "shift":
            y += t["x"] * torch.as_tensor(_shifts(case, seed).astype(np.float32 if single else np.float64), device=DEV)
        y = case["alpha"] * y + (case["beta"] * t["y"] if case["beta"] else 0.0)
        return [y, (y * y).sum(0).cpu().numpy(), (t["x"] * y).sum(0).cpu().numpy()] if op == "dots" else y
    s = torch.as_tensor(_shifts(case, seed), device=DEV)
    if op == "minres":
        x, rel = _exact_minres(ell, s, t["b"], case["iters"])
        return [x, None, rel.cpu().numpy()]
    x, rel = _exact_gmres(ell, s, t["b"], case["iters"])
    return [x, None, rel.numpy()]
