"""The work that programs have this library do, as a list of cases that can be timed and checked.

A case is a scene (or a batch of scenes) of rectangular air domains with 50-cell absorbing layers, a number of time
steps and what the program reads back: the receiver series and the pressure frames of the air domains.

    listed()              the cases
    draw(rng)             one more case of the same ranges
    prepare(case, seed)   the solver a program holds, with the state of `seed` loaded
    run(state)            one pass: advance the solver, read the series and the frames
    work(case)            bytes and floating-point operations of one pass
    exact(case, seed)     what run() returns for a new state, in 64 bits

exact() is a solver of its own in torch and numpy, double precision, for the scenes used here: domains that meet along
whole edges.  It knows openPSTD's rules for the absorbing layers and for the order of vertical neighbours.
"""
import math

import numpy as np
import torch

from openpstd_amd import BatchSolver, PSTDConfiguration, PSTDKernel, RecordingCallback
from openpstd_amd import abi_types
from openpstd_amd import workloads

PML_CELLS = 50
MODES = 16  # standing waves summed into a loaded field


def _case(name, cols, rows, steps, **more):
    c = {"name": name, "shape": "grid", "cols": cols, "rows": rows, "scenes": 1, "steps": steps, "form": "fft",
         "receivers": 4, "spectral": False, "walls": "open", "patch": 70, "speakers": 0, "call": "advance",
         "save_nth": 0, "state": False}
    c.update(more)
    return c


def listed():
    return [
        # an interactive view of a small room: one step, then the frame that is shown (the smallest call)
        _case("room_step", "100", "50", 1, receivers=1, speakers=1),
        # the same room for longer, its whole state read back as for a checkpoint
        _case("room_checkpoint", "100", "50", 40, receivers=1, speakers=1, state=True),
        # kernel.run(): the call of the command line, set-up and frame callbacks included
        _case("lshape_run", "256,256", "128,128", 121, shape="lshape", walls="mixed", speakers=3, call="run", save_nth=40),
        # the L-shape with receivers between the cells (spectral interpolation after every step)
        _case("lshape_spectral", "256,256", "128,128", 40, shape="lshape", walls="mixed", receivers=10, spectral=True),
        # three rooms in a row, odd sides, partly reflecting walls, another window length
        _case("rooms_odd", "333,141,477", "217", 40, walls="drawn", patch=60),
        # one ordinary hall, line lengths just past a power of two
        _case("square1024", "1024", "1024", 20, receivers=8),
        # the same hall in the BF16 matrix form
        _case("square1024_bf16", "1024", "1024", 20, receivers=8, form="gemm_bf16"),
        # a wide ragged site: 4096-point rows, 2048-point columns
        _case("site_2501x1237", "2501", "1237", 10, receivers=16, walls="drawn"),
        # the largest single domain in use: 8192-point lines
        _case("square4096", "4096", "4096", 10, receivers=16),
        # a parameter study: different scenes advanced together
        _case("batch", "64", "600", 20, shape="batch", scenes=12, receivers=1, walls="drawn"),
        # many source positions of one geometry advanced together, in the FFT and the FP16 matrix form
        _case("sources_fft", "512,512", "1024", 10, scenes=16, receivers=8),
        _case("sources_f16", "512,512", "1024", 10, scenes=16, receivers=8, form="gemm_f16"),
    ]


def _window(patch):
    return 2 * int(math.floor((np.float32(patch) * 0.7 - 17) / 2.0 + 0.5))


def _side(rng, lo, hi, patch):
    """A side in [lo, hi], spread over its logarithm; n + 2w a power of two is refused by the library."""
    w = _window(patch)
    while True:
        n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        if (n + 2 * w) & (n + 2 * w - 1):
            return n


def draw(rng):
    kind = rng.choice(["single", "single", "single", "row", "column", "grid", "lshape", "batch", "sources", "sources"])
    patch = rng.choice([70, 70, 70, 60, 50])
    form = rng.choice(["fft", "fft", "fft", "gemm_f16", "gemm_bf16"])
    side = lambda lo, hi: _side(rng, lo, hi, patch)  # noqa: E731
    walls = rng.choice(["open", "drawn", "mixed"])
    if kind == "single":
        c = _case("", str(side(64, 4096)), str(side(64, 4096)), 0, walls=walls)
    elif kind == "row":
        c = _case("", ",".join(str(side(64, 1024)) for _ in range(rng.randint(2, 4))), str(side(64, 1024)), 0, walls=walls)
    elif kind == "column":
        c = _case("", str(side(64, 1024)), ",".join(str(side(64, 1024)) for _ in range(rng.randint(2, 4))), 0, walls=walls)
    elif kind in ("grid", "lshape"):
        c = _case("", "%d,%d" % (side(64, 700), side(64, 700)), "%d,%d" % (side(64, 700), side(64, 700)), 0, shape=kind,
                  walls=walls)
    elif kind == "batch":
        patch = 70  # batch sides avoid the lengths refused with this window
        c = _case("", str(rng.randint(64, 100)), str(rng.randint(200, 700)), 0, shape="batch", scenes=rng.randint(2, 14),
                  walls="drawn", receivers=1)
    else:
        c = _case("", "%d,%d" % (side(128, 512), side(128, 512)), str(side(256, 1024)), 0, scenes=rng.randint(2, 16),
                  receivers=8)
    c.update(form=form, patch=patch)
    c["steps"] = int(round(math.exp(rng.uniform(0, math.log(60)))))
    if c["shape"] != "batch":
        cells = sum(w * h for _, _, w, h in _rects(c, 0)) * c["scenes"]
        c["steps"] = max(1, min(c["steps"], int(1.5e8 / cells)))
        if c["scenes"] == 1:
            c["receivers"] = rng.randint(1, 16)
            c["spectral"] = cells < 1e6 and rng.random() < 0.25
            c["speakers"] = rng.choice([0, 0, 1]) * len(_rects(c, 0))
            if cells < 2e5 and rng.random() < 0.3:
                c.update(call="run", speakers=len(_rects(c, 0)), spectral=False,
                         form="fft", save_nth=max(1, c["steps"] // rng.randint(1, 4)))
    del c["name"]
    return c


# ------------------------------------------------------------------ scenes


def _rects(case, scene):
    """Air domains (x, y, nx, ny) of one scene, in cells."""
    if case["shape"] == "batch":
        # one to four domains in a row, a column or a grid, sides between the two numbers of the case
        rng = np.random.RandomState(1000 + scene)
        lo, hi = int(case["cols"]), int(case["rows"])

        def side():
            while True:
                n = int(rng.randint(lo, hi + 1))
                if n not in workloads.EXCLUDED_SIDES:
                    return n

        kind = rng.randint(4)
        cols = [side() for _ in range((1, rng.randint(2, 5), 1, 2)[kind])]
        rows = [side() for _ in range((1, 1, rng.randint(2, 5), 2)[kind])]
    else:
        cols = [int(v) for v in case["cols"].split(",")]
        rows = [int(v) for v in case["rows"].split(",")]
    out = []
    for j, h in enumerate(rows):
        for i, w in enumerate(cols):
            if not (case["shape"] == "lshape" and i == 1 and j == 1):
                out.append((sum(cols[:i]), sum(rows[:j]), w, h))
    return out


def _absorption(case, scene, n):
    """Absorption of every air domain's edges T, L, B, R: part of the geometry, the same for every seed."""
    rng = np.random.RandomState(7 + scene)
    if case["walls"] == "open":
        return [[1.0] * 4] * n
    if case["walls"] == "mixed":
        return [[(0.0, 0.5, 1.0)[rng.randint(3)] for _ in range(4)] for _ in range(n)]
    return [[float(np.float32(rng.uniform(0.05, 1))) for _ in range(4)] for _ in range(n)]


def _points(case, scene, seed):
    """Speakers and receivers in cells; receivers stay two cells away from the edges."""
    rng = np.random.RandomState([seed % (1 << 31), scene])
    rects = _rects(case, scene)
    speakers = []
    for k in range(case["speakers"]):
        x, y, w, h = rects[k % len(rects)]
        speakers.append((x + rng.randint(8, w - 8) + 0.5, y + rng.randint(8, h - 8) + 0.5))
    receivers = []
    for _ in range(case["receivers"]):
        x, y, w, h = rects[rng.randint(len(rects))]
        f = rng.randint(1, 8, 2) / 8.0 if case["spectral"] else (0.25, 0.25)
        receivers.append((x + rng.randint(2, w - 2) + float(f[0]), y + rng.randint(2, h - 2) + float(f[1])))
    return speakers, receivers


def _loaded(case, scene, seed):
    """The state a program continues from: for every air domain p0, px0, py0, vx0 and vy0 (float32), a sum of standing
    waves of at least 5 cells' length; zero in the absorbing layers.  None: the scene starts from its speakers."""
    if case["speakers"]:
        return None
    out = []
    for d, (_, _, w, h) in enumerate(_rects(case, scene)):
        rng = np.random.RandomState([seed % (1 << 31), scene, d, 17])

        def waves(ny, nx):
            kx, ky = rng.uniform(0, 2 * np.pi / 5, (2, MODES))
            fx, fy = rng.uniform(0, 2 * np.pi, (2, MODES))
            a = rng.uniform(-1, 1, MODES) / 4
            up, across = np.cos(np.outer(np.arange(ny), ky) + fy), np.cos(np.outer(np.arange(nx), kx) + fx)
            return ((a * up) @ across.T).astype(np.float32)

        px, py = waves(h, w), waves(h, w)
        imp = np.float32(1.0 / 408.0)  # velocities are pressures over rho c
        out.append({"p0": px + py, "px0": px, "py0": py, "vx0": waves(h, w + 1) * imp, "vy0": waves(h + 1, w) * imp})
    return out


def _configuration(case, scene, seed):
    conf = PSTDConfiguration()
    workloads.base_settings(conf, case["steps"])
    conf.Settings.SetPatchError(float(case["patch"]))
    if case["save_nth"]:
        conf.Settings.SetSaveNth(case["save_nth"])
    rects = _rects(case, scene)
    for (x, y, w, h), a in zip(rects, _absorption(case, scene, len(rects))):
        conf.Domains.append(workloads.domain(x, y, w, h, dict(zip("TLBR", a))))
    speakers, receivers = _points(case, scene, seed)
    conf.Speakers += [(workloads._world_pos(x), workloads._world_pos(y), 0.0) for x, y in speakers]
    conf.Receivers += [(workloads._world_pos(x), workloads._world_pos(y), 0.0) for x, y in receivers]
    if case["spectral"]:
        conf.receiver_mode = abi_types.PSTD_RECEIVER_SPECTRAL
    return conf


# ------------------------------------------------------------------ the calls


def prepare(case, seed):
    state = {"case": case, "domains": [len(_rects(case, s)) for s in range(case["scenes"])]}
    confs = [_configuration(case, s, seed) for s in range(case["scenes"])]
    if case["scenes"] > 1:
        solver = state["solver"] = BatchSolver(confs, form=case["form"])
        for s in range(case["scenes"]):
            for d, fields in enumerate(_loaded(case, s, seed) or []):
                for name, values in fields.items():
                    solver.set_field(s, d, name, values)
        return state
    kernel = state["kernel"] = PSTDKernel(GPU=True)
    kernel.initialize_kernel(confs[0])
    kernel.set_form(case["form"])
    if case["call"] == "run":
        return state
    solver = state["solver"] = kernel.prepare()
    for d, fields in enumerate(_loaded(case, 0, seed) or []):
        for name, values in fields.items():
            solver.set_field(d, name, values)
    return state


def run(state):
    case = state["case"]
    if case["call"] == "run":
        got = RecordingCallback()
        state["kernel"].run(got)
        series = [[v for _, v in got.samples[r]] for r in sorted(got.samples)]
        return {"frames": [f for _, _, f in got.frames], "samples": np.array(series, dtype=np.float32)}
    solver = state["solver"]
    samples = solver.advance(case["steps"])
    if case["scenes"] > 1:
        frames = [solver.field(s, d, "p0") for s, n in enumerate(state["domains"]) for d in range(n)]
    else:
        frames = [solver.field(d, "p0") for d in range(state["domains"][0])]
    out = {"frames": frames, "samples": samples}
    if case["state"]:
        out["state"] = {name: [solver.field(d, name) for d in range(state["domains"][0])]
                        for name in ("px0", "py0", "vx0", "vy0")}
    return out


def work(case):
    """48 bytes per cell and Runge-Kutta stage (p0, vx, vy of the stage before and the four fields at t_n read, five
    fields written), the frames once; two real transforms and the filter per line and derivative."""
    cells = air = flops = 0.0
    for s in range(case["scenes"]):
        scene = _Scene(case, s)
        air += sum(w * h for _, _, w, h in _rects(case, s))
        for d in scene.domains:
            if d.rigid:
                continue
            cells += d.nx * d.ny
            for lines, n in ((d.ny, d.nx), (d.nx, d.ny)):
                f = scene.length(n)
                flops += 2 * lines * (2 * 2.5 * f * math.log2(f) + 3 * f + 2 * n)
    return {"bytes": case["steps"] * 6 * 48 * cells + 4 * air, "flops": case["steps"] * 6 * flops}


# ------------------------------------------------------------------ the same in 64 bits

LEFT, RIGHT, TOP, BOTTOM = range(4)
OPPOSITE = (RIGHT, LEFT, BOTTOM, TOP)


class _Domain:
    def __init__(self, alpha, x, y, nx, ny, rho, parents=(), secondary=False):
        self.x, self.y, self.nx, self.ny, self.alpha = x, y, nx, ny, alpha
        root = np.sqrt(np.float32(1) - np.float32(alpha))
        with np.errstate(divide="ignore"):
            impedance = -((root + np.float32(1)) / (root - np.float32(1)))
        self.rigid = bool(impedance > 1000)
        self.rho = 1e30 if self.rigid else float(np.float32(rho) * impedance)
        self.parents, self.secondary, self.pml = list(parents), secondary, bool(parents)
        self.nb = [None] * 4


def _meet(a, b):
    """The side of `a` on which `b` lies, or None."""
    over_y = max(a.y, b.y) < min(a.y + a.ny, b.y + b.ny)
    over_x = max(a.x, b.x) < min(a.x + a.nx, b.x + b.nx)
    if a.x + a.nx == b.x:
        return RIGHT if over_y else None
    if a.x == b.x + b.nx:
        return LEFT if over_y else None
    if a.y + a.ny == b.y:
        return BOTTOM if over_x else None
    if a.y == b.y + b.ny:
        return TOP if over_x else None
    return None


class _Scene:
    """The domains of one scene with their absorbing layers, and the time step, in 64 bits."""

    def __init__(self, case, scene):
        s = PSTDConfiguration().Settings
        self.dx = float(np.float32(workloads.DX))
        self.c1, self.rho = 340.0, float(np.float32(1.2))
        self.dt = float(np.float32(np.float32(np.float32(0.5) * np.float32(self.dx)) / np.float32(self.c1)))
        self.alphas = [float(np.float32(a)) for a in s.GetRKCoefficients()]
        self.patch, self.w = case["patch"], _window(case["patch"])
        rects = _rects(case, scene)
        self.domains, corners = [], []
        for r in rects:
            self._add(_Domain(1.0, *r, self.rho))
        strips = []
        for d, (t, l, b, r) in zip(list(self.domains), _absorption(case, scene, len(rects))):
            walls = {LEFT: l, RIGHT: r, TOP: b, BOTTOM: t}  # openPSTD exchanges top and bottom
            order = (LEFT, TOP, RIGHT, BOTTOM)
            for i, side in enumerate(order):
                if d.nb[side] is not None:
                    continue
                n = PML_CELLS
                x, y, nx, ny = {LEFT: (d.x - n, d.y, n, d.ny), RIGHT: (d.x + d.nx, d.y, n, d.ny),
                                TOP: (d.x, d.y - n, d.nx, n), BOTTOM: (d.x, d.y + d.ny, d.nx, n)}[side]
                strip = _Domain(max(walls[side], 1e-5), x, y, nx, ny, self.rho, [d])
                strips.append(strip)
                if walls[side] <= 0:
                    continue
                for k in ((i + 1) % 4, (i + 3) % 4):
                    cs = order[k]
                    ox = {LEFT: -n, RIGHT: nx}.get(cs, 0)
                    oy = {TOP: -n, BOTTOM: ny}.get(cs, 0)
                    alpha = min(max(1e-5, walls[cs]), strip.alpha)
                    corners.append((_Domain(alpha, x + ox, y + oy, n, n, self.rho, [strip], True), cs))
        for p in strips:
            self._add(p)
        places = {}
        for c, cs in corners:
            if c.parents[0].nb[cs] is None:
                places.setdefault((c.x, c.y), []).append(c)
        for key in sorted(places):
            kept = []
            for c in places[key]:
                user = c.parents[0].parents[0]
                twin = next((k for k in kept if len(k.parents) == 1 and k.parents[0].parents[0] is user), None)
                if twin is None:
                    kept.append(c)
                else:
                    twin.parents += c.parents
            for c in kept:
                self._add(c)
        for d in self.domains:
            if d.pml:
                self._attenuation(d)

    def _add(self, d):
        for o in self.domains:
            if d.secondary and o.secondary or d.secondary and not o.pml or o.secondary and not d.pml:
                continue
            if d.pml and o.pml and not (d.secondary and o in d.parents or o.secondary and d in o.parents):
                if len(o.parents) != 1 or len(d.parents) != 1 or d.parents[0] not in o.parents[0].nb:
                    continue
            side = _meet(d, o)
            if side is None or o.pml and not d.pml and d not in o.parents or d.pml and not o.pml and o not in d.parents:
                continue
            assert d.nb[side] is None and o.nb[OPPOSITE[side]] is None, "domains meet along whole edges"
            d.nb[side], o.nb[OPPOSITE[side]] = o, d
        self.domains.append(d)

    def _attenuation(self, d):
        n, rho, amp = PML_CELLS, self.rho, 20000.0
        air = lambda s: d.nb[s] is not None and not d.nb[s].pml  # noqa: E731
        if d.secondary and sum(v is not None for v in d.nb) == 2:
            along = {"x": d.nb[LEFT] is not None, "y": d.nb[BOTTOM] is not None}
        elif d.secondary:
            along = {"x" if d.nb[LEFT] or d.nb[RIGHT] else "y": d.nb[LEFT] is not None or d.nb[BOTTOM] is not None}
        else:
            along = {"x" if air(LEFT) or air(RIGHT) else "y": air(LEFT) or air(BOTTOM)}
        one = torch.ones
        d.damp = {"px": one(1, 1), "py": one(1, 1), "vx": one(1, 1), "vy": one(1, 1)}
        for axis, rising in along.items():
            p = np.exp(-amp * ((np.arange(n) + 0.5) / n) ** 4 * self.dt / rho)
            v = np.exp(-rho * amp * (np.arange(n + 1) / n) ** 4 * self.dt)
            for name, f in (("p" + axis, p), ("v" + axis, v)):
                f = torch.from_numpy((f if rising else f[::-1]).copy())
                d.damp[name] = f[None, :] if axis == "x" else f[:, None]

    def window(self, n):
        w = self.w
        while w > n:
            w //= 2
        return w

    def length(self, n):
        return 1 << (n + 2 * self.window(n)).bit_length()

    def line(self, d, axis, vel, main, side1, side2, delta=None):
        """The spectral derivative (or, with `delta`, the shift by delta cells) along the last dimension of `main`; side1
        and side2 are the neighbours' lines or None."""
        n = d.nx if axis == "x" else d.ny
        w, nm = self.window(n), main.shape[-1]
        F = self.length(n)
        o1, o2 = (d.nb[LEFT], d.nb[RIGHT]) if axis == "x" else (d.nb[BOTTOM], d.nb[TOP])
        coef = []
        for o in (o1, o2):
            z = (o.rho if o else d.rho) / d.rho
            r = (z - 1) / (z + 1)
            coef.append((2 * z / (z + 1), -r) if vel else (2 / z / (1 / z + 1), r))
        xs = (np.arange(2 * w + 1) - w) / w
        win = torch.from_numpy(np.exp(-math.log(10.0) * ((self.patch - 40) / 20.0 + 1) * xs ** 6)).to(main.device)
        buf = torch.zeros(main.shape[:-1] + (F,), dtype=torch.float64, device=main.device)
        buf[..., w:w + nm] = main
        head, tail = main[..., vel:w + vel].flip(-1), main[..., nm - w - vel:nm - vel].flip(-1)
        if side1 is not None:
            buf[..., :w] = coef[0][0] * side1[..., side1.shape[-1] - w - vel:side1.shape[-1] - vel]
            buf[..., w + nm:2 * w + nm] = 0
        buf[..., :w] = (buf[..., :w] + coef[0][1] * head) * win[:w]
        right = coef[1][1] * tail
        if side2 is not None:
            right = right + coef[1][0] * side2[..., vel:w + vel]
        buf[..., w + nm:2 * w + nm] = right * win[w + 1:]
        m = np.arange(F // 2 + 1)
        if delta is None:
            k = m * (math.pi / self.dx) / (F // 2)
            h = np.exp((1j if vel else -1j) * k * self.dx * 0.5) * 1j * k
            h[0] = 0
        else:
            h = np.exp(1j * math.pi * m * delta / (F // 2))
        h[-1] = h[-1].real
        out = torch.fft.irfft(torch.fft.rfft(buf) * torch.from_numpy(h).to(main.device), n=F)
        return out[..., w:w + (n if vel or delta is not None else n + 1)]

    def stage(self, now, s):
        """One Runge-Kutta stage: the four fields of every domain from `now` (p, vx, vy) and the state at t_n."""
        new = {}
        for d in self.domains:
            u = dict(d.tn)
            if not d.rigid:
                def L(axis, vel, name):
                    turn = (lambda a: a) if axis == "x" else (lambda a: a.T)
                    o1, o2 = (d.nb[LEFT], d.nb[RIGHT]) if axis == "x" else (d.nb[BOTTOM], d.nb[TOP])
                    s1, s2 = (turn(now[o][name]) if o else None for o in (o1, o2))
                    return turn(self.line(d, axis, vel, turn(now[d][name]), s1, s2))

                cv, cp = s / d.rho, s * d.rho * self.c1 ** 2
                u["vx"] = d.tn["vx"] - cv * L("x", 0, "p")
                u["vy"] = d.tn["vy"] - cv * L("y", 0, "p")
                u["px"] = d.tn["px"] - cp * L("x", 1, "vx")
                u["py"] = d.tn["py"] - cp * L("y", 1, "vy")
            new[d] = u
        for u in new.values():
            u["p"] = u["px"] + u["py"]
        return new

    def step(self, p):
        now = {d: {"p": p[d], "vx": d.tn["vx"], "vy": d.tn["vy"]} for d in self.domains}
        for a in self.alphas:
            now = self.stage(now, self.dt * a)
        for d in self.domains:
            d.tn = {k: now[d][k] * d.damp[k] if d.pml else now[d][k] for k in ("px", "py", "vx", "vy")}
        return {d: now[d]["p"] for d in self.domains}

    def sample(self, p, x, y, spectral):
        d = next(d for d in reversed(self.domains) if not d.pml and d.x <= x <= d.x + d.nx and d.y <= y <= d.y + d.ny)
        cx, cy = int(x) - d.x, int(y) - d.y
        if not spectral:
            return p[d][cy, cx]
        side = lambda o, s: p[o.nb[s]] if o.nb[s] is not None else None  # noqa: E731

        def column(o, rows):
            cut = lambda a: None if a is None else a[rows]  # noqa: E731
            return self.line(o, "x", 0, p[o][rows], cut(side(o, LEFT)), cut(side(o, RIGHT)), x - int(x))[:, cx]

        o1, o2, w = d.nb[BOTTOM], d.nb[TOP], self.window(d.ny)
        first = column(o1, slice(o1.ny - w, o1.ny)) if o1 is not None else None
        last = column(o2, slice(0, w)) if o2 is not None else None
        return self.line(d, "y", 0, column(d, slice(0, d.ny)), first, last, y - int(y))[cy]


def exact(case, seed):
    device = "cuda" if torch.cuda.is_available() else "cpu"
    if sum(w * h for s in range(case["scenes"]) for _, _, w, h in _rects(case, s)) * case["steps"] > 2e7 and device == "cpu":
        return None  # minutes
    frames, series, last = [], [], None
    for s in range(case["scenes"]):
        scene = _Scene(case, s)
        put = lambda a: torch.as_tensor(np.asarray(a, dtype=np.float64), device=device)  # noqa: E731
        speakers, receivers = _points(case, s, seed)
        loaded, p = _loaded(case, s, seed), {}
        for i, d in enumerate(scene.domains):
            if d.pml:
                d.damp = {k: v.to(device).double() for k, v in d.damp.items()}
            shapes = {"px": (d.ny, d.nx), "py": (d.ny, d.nx), "vx": (d.ny, d.nx + 1), "vy": (d.ny + 1, d.nx)}
            d.tn = {k: torch.zeros(v, dtype=torch.float64, device=device) for k, v in shapes.items()}
            p[d] = torch.zeros(d.ny, d.nx, dtype=torch.float64, device=device)
            if loaded is not None and not d.pml:
                d.tn = {k: put(loaded[i][k + "0"]) for k in shapes}
                p[d] = put(loaded[i]["p0"])
            for x, y in speakers:
                beta = float(np.float32(3e-6 * float(np.float32(340.0 / scene.dx)) ** 2))
                ax = x - 0.5 - d.x - np.arange(d.nx)[None, :]
                ay = y - 0.5 - d.y - np.arange(d.ny)[:, None]
                g = np.exp(-beta * scene.dx ** 2 * (ax ** 2 + ay ** 2))
                angle = np.arctan2(ax, ay)
                p[d] += put(g)
                d.tn["px"] += put(np.cos(angle) ** 2 * g)
                d.tn["py"] += put(np.sin(angle) ** 2 * g)
        steps = []
        for t in range(case["steps"]):
            p = scene.step(p)
            if case["call"] != "run" or t % case["save_nth"] == 0:
                steps.append(torch.stack([scene.sample(p, x, y, case["spectral"]) for x, y in receivers]))
                if case["call"] == "run":
                    frames += [p[d].reshape(-1).cpu() for d in scene.domains if not d.pml]
        series.append(torch.stack(steps).cpu())
        if case["call"] != "run":
            frames += [p[d].cpu() for d in scene.domains if not d.pml]
        last = scene
    samples = torch.cat(series, 1)
    out = {"frames": frames, "samples": samples.T.contiguous() if case["call"] == "run" else samples}
    if case["state"]:
        out["state"] = {k + "0": [d.tn[k].cpu() for d in last.domains if not d.pml] for k in ("px", "py", "vx", "vy")}
    return out
