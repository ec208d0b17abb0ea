"""The lower-order part of an RCCSDT iteration in few launches, for one engine or an ensemble.

The programs of RCCSDTEngine (T1 dressing, singles/doubles residual, T2-dressed intermediates) are lists of
contractions and strided copies that accumulate into some twenty tensors.  Issued one by one they are some
150 launches of 5 to 8 us each, most of an iteration of a small molecule (nocc=5, nvir=8: 1.01 ms, 0.43 ms this
way; nocc=5, nvir=19: 1.32 and 0.70 ms; nocc=8, nvir=38: 5.60 and 5.22 ms).  Here every contraction writes its
own partial result, so all of a program whose operands are known run side by side: the small ones as one
grouped launch (dcc_contract_grouped_f64), the large ones on their own, and one dcc_combine launch then sums
the partials and copies of every tensor of that stage, in the order of the program.  In an ensemble a grouped
launch takes the same contraction of every system.  Divisions by the
denominators, the amplitude update and the T3 terms ride along as further terms of those sums; dot products
are one launch of many (dcc_dots_f64). 
"""
import itertools

import numpy as np

from distr_cc import _lib as L
from distr_cc.batched import _GroupedPhase
from distr_cc.device import DeviceArray, mem_get_info
from distr_cc.t3_engine import GemmLaunch, LIBRARY_TILE, Operand, plan_einsum, upload_tables

# 64x64 tiles below which a contraction does not fill the chip and joins its stage's grouped launch
SMALL_TILES = 64
# partials of one engine above which it keeps the one-by-one programs: an iteration of that size is bound by
# the contractions and the extra pass over the partials only costs (nocc=10, nvir=90, 0.9 GB of partials:
# 179.6 ms against 178.1)
MAX_PARTIAL_BYTES = 512 << 20


def term(op, letters, coef=1.0, count=1, cstride=0):
    """A source of a combination: the Operand ``op`` over the target's ``letters``, ``count`` slices apart by
    ``cstride`` elements summed up."""
    return (op.buf.ptr + op.base * op.buf.dtype.itemsize, [op.strides.get(x, 0) for x in letters], float(coef),
            int(count), int(cstride), int(op.buf.dtype == np.float32))


class Combine:
    """One dcc_combine launch.  Jobs: (target Operand, letters, extents, terms, options), options beta, acc
    (DeviceArray), eia (DeviceArray) and rank."""

    def __init__(self, jobs):
        rows, terms, begin = [], [], 0
        for dst, letters, shape, ts, opt in jobs:
            pad = 4 - len(letters)
            total = int(np.prod(shape))
            if total >= 1 << 31:
                raise ValueError("combination of more than 2^31 elements")
            if total == 0:
                continue
            rows.append((dst.buf.ptr + dst.base * dst.buf.dtype.itemsize, [1] * pad + list(shape),
                         [0] * pad + [dst.strides[x] for x in letters], opt.get("beta", 0.0),
                         opt["acc"].ptr if "acc" in opt else 0, opt["eia"].ptr if "eia" in opt else 0,
                         opt.get("rank", 0), len(terms), len(ts), begin, int(dst.buf.dtype == np.float32)))
            terms += [(ptr, [0] * pad + st, c, n, cs, f) for ptr, st, c, n, cs, f in ts]
            begin += -(-total // 1024)
        self.njobs, self.nwg = len(rows), begin
        self.jobs = DeviceArray.from_host(_table(rows, L.COMBINE_DTYPE))
        self.terms = DeviceArray.from_host(_table(terms, L.TERM_DTYPE))

    def run(self, stream):
        L.call("dcc_combine", self.jobs.vp, self.terms.vp, self.njobs, self.nwg,
               stream.handle if stream is not None else None)


class Dots:
    """One dcc_dots_f64 launch.  Jobs: (x, y, u or None, out pointer, n, nocc, nvir)."""

    def __init__(self, jobs):
        self.jobs = DeviceArray.from_host(_table([(x.ptr, y.ptr, u.ptr if u is not None else 0, out, n, o, v)
                                                  for x, y, u, out, n, o, v in jobs], L.DOT_DTYPE))
        self.n = len(jobs)
        self.partials = DeviceArray((self.n * int(L._lib.dcc_dots_partials()),))

    def run(self, stream):
        L.call("dcc_dots_f64", self.jobs.vp, self.n, self.partials.vp, stream.handle if stream is not None else None)


def _table(rows, dtype):
    arr = np.zeros(max(len(rows), 1), dtype=dtype)
    for n, r in enumerate(rows):
        arr[n] = tuple(r)
    return arr


class Step:
    """A device action of one engine (run(stream))."""

    def __init__(self, fn):
        self.run = fn


class NotSchedulable(ValueError):
    """A program whose operations cannot run stage by stage."""


def _need(ok, why):
    if not ok:
        raise NotSchedulable("program cannot be scheduled: " + why)


def _small(g):
    M, N = g.args[:2]
    return -(-M // 64) * -(-N // 64) * g.nbatch <= SMALL_TILES


class _Partials:
    """Partial results of one phase of one engine: sized first, then views of the engine's arena."""

    def __init__(self):
        self.used = 0

    def size(self, op):
        """Reserve room for a tensor shaped and ordered as the operand ``op``; returns its offset."""
        off = self.used
        self.used += -(-int(np.prod(op.shape)) // 2) * 2    # pairs stay aligned
        return off


class LowerSchedule:
    """Launch lists of the phases "dress", "r1r2", "update12" and "imds3" for ``engines`` (RCCSDTEngine) on one
    stream.  ``grouped`` holds the grouped launches (for the tile autotuner of an ensemble)."""

    def __init__(self, engines, stream):
        self.engines, self.stream = engines, stream
        self.grouped = []
        targets = {name: [self._targets(e, name) for e in engines] for name in ("r1r2", "imds3")}
        arenas = []
        for k, e in enumerate(engines):
            need = max(t[k][1].used for t in targets.values())
            arenas.append(DeviceArray((max(need, 1),)))
        self.arenas = arenas
        self.phases = {"dress": self._plan_dress(), "r1r2": self._plan_program("r1r2", targets["r1r2"]),
                       "update12": self._plan_update(), "imds3": self._plan_program("imds3", targets["imds3"])}

    @staticmethod
    def fits(engines):
        """Whether the lower-order part of every engine is worth and able to run this way: FP64 triples, one chunk
        of Z, partials within MAX_PARTIAL_BYTES, tensors below 2^31 elements; and whether the partials of all of
        them leave as much of the device's free memory as they take (the one-by-one programs need next to none, so
        an ensemble that fills the device runs on those)."""
        total = 0
        for e in engines:
            if e.mixed or len(e.tr._lower["chunks"]) != 1 or e.nmo ** 4 >= 1 << 31:
                return False
            try:
                used = 8 * max(LowerSchedule._targets(e, n)[1].used for n in ("r1r2", "imds3"))
            except NotSchedulable:
                return False
            if used > MAX_PARTIAL_BYTES:
                return False
            total += used + 8 * (e.nocc * e.nvir) ** 2    # and the E_ooov partial of _plan_update
        return 2 * total <= mem_get_info()[0]

    # ------------------------------------------------------------------ programs
    @staticmethod
    def _targets(eng, name):
        """The tensors a program accumulates into, in order: {id(buffer): [Operand, letters, level, parts]} with
        parts ("ein", offset of the partial, op, stage) or ("src", op); and the partials' sizes.  A tensor's stage is
        known when it is read, so every contribution to it must come before."""
        out, part, read = {}, _Partials(), set()

        def level(op):
            read.add(id(op.buf))
            return out[id(op.buf)][2] if id(op.buf) in out else 0

        for op in eng.prog[name].ops:
            _need(op[0] in ("axpby", "ein"), "a step that is no contraction or copy")
            dst = op[1] if op[0] == "axpby" else op[5]
            if op[0] == "axpby":
                _, _, src, letters, alpha, beta = op
                _need(sorted(letters) == sorted(dst.letters), "a copy that broadcasts into its target")
                if beta == 0.0:
                    _need(id(dst.buf) not in out and dst.shape is not None, "a tensor that is set twice")
                    out[id(dst.buf)] = [dst, dst.letters, 0, []]
                at, entry = level(src), ("src", op)
            else:
                _, _, sub, A, B, C, alpha, beta = op
                at = max(level(A), level(B))
            t = out.get(id(dst.buf))
            _need(t is not None, "an accumulation into a tensor that is not set first")
            _need(id(dst.buf) not in read, "a tensor that is read before its last contribution")
            if op[0] == "ein":
                _need(C.strides == t[0].strides and C.base == t[0].base and beta == 1.0, "a contraction into a view")
                entry = ("ein", part.size(t[0]), op, at)
            t[2] = max(t[2], at + 1)
            t[3].append(entry)
        return out, part

    def _plan_program(self, name, targets):
        """Per stage: the contractions whose operands are complete, then the tensors of the next level."""
        levels = max(t[2] for out, _ in targets for t in out.values())
        gemms = [[] for _ in range(levels)]
        jobs = [[] for _ in range(levels)]
        for k, (eng, (out, _)) in enumerate(zip(self.engines, targets)):
            for dst, letters, lev, parts in out.values():
                shape, terms = [eng.ext[x] for x in letters], []
                for p in parts:
                    if p[0] == "src":
                        terms.append(term(p[1][2], letters, p[1][4]))
                    else:
                        _, off, (_, nm, sub, A, B, C, alpha, _b), stage = p
                        P = DeviceArray(dst.shape, np.float64, ptr=self.arenas[k].ptr + 8 * off, owner=False)
                        g = plan_einsum(nm, sub, A, B, Operand(P, letters, dst.shape), alpha, 0.0, eng.ext,
                                        [({}, {}, {})])
                        gemms[stage].append((k, g))
                        terms.append(term(Operand(P, letters, dst.shape), letters))
                terms += self._t3_terms(eng, dst, letters) if name == "imds3" else []
                jobs[lev - 1].append((dst, letters, shape, terms, {}))
        steps = []
        upload_tables([g for st in gemms for _, g in st])
        for stage in range(levels):
            steps += self._contractions(gemms[stage])
            steps.append(Combine(jobs[stage]))
        return steps

    def _t3_terms(self, eng, dst, letters):
        """The T3 terms of W_vooo and W_vvvo (rccsdt.py:323-366), computed by the update12 phase."""
        lo, o, v = eng.tr._lower, eng.nocc, eng.nvir
        if dst.buf is eng.imd["W_oovo"]:
            return [term(Operand(lo["P3"], letters, (o, o, v, o)), letters, 1.0, o, o * o * v * o)]
        if dst.buf is eng.imd["W_ovvv"]:
            return [term(Operand(lo["dWovvv"], letters, (o, v, v, v)), letters)]
        return []

    def _contractions(self, gemms):
        """Launches of independent contractions [(engine, GemmLaunch)].  One engine: the small ones together,
        a large one alone.  An ensemble: the n-th of every engine that has so many together, which fills the chip
        already."""
        if len(self.engines) == 1:
            small = [g for _, g in gemms if _small(g)]
            steps = [small[0]] if len(small) == 1 else [self._group(small, True)] if small else []
            return steps + [g for _, g in gemms if not _small(g)]
        per = {}
        for k, g in gemms:
            per.setdefault(k, []).append(g)
        return [self._group([g for g in gs if g is not None], False) for gs in itertools.zip_longest(*per.values())]

    def _group(self, launches, small):
        ph = _GroupedPhase(launches, small)
        ph.prepare(LIBRARY_TILE, self.stream)
        self.grouped.append(ph)
        return ph

    # -------------------------------------------------------------------- phases
    def _plan_dress(self):
        """T1 dressing (RCCSDTEngine "dress"): G and the Fock matrix are transformed in place, one index after
        the other; the two-electron part of the Fock matrix is a sum over strided views of G."""
        first, last, chain = [], [], [[] for _ in range(4)]
        for k, e in enumerate(self.engines):
            n, o = e.nmo, e.nocc
            nv = lambda b, l: Operand(b, l, b.shape)
            first += [(nv(e.G, "PQRS"), "PQRS", [n] * 4, [term(nv(e.G0, "PQRS"), "PQRS")], {}),
                      (nv(e.Fd, "PQ"), "PQ", [n] * 2, [term(nv(e.Hc, "PQ"), "PQ")], {})]
            eins = [op for op in e.prog["dress"].ops if op[0] == "ein" and not op[1].startswith("jk")]
            plan = lambda op: plan_einsum(op[1], op[2], op[3], op[4], op[5], op[6], op[7], e.ext, [({}, {}, {})])
            by = {op[1]: op for op in eins}
            for q, names in enumerate((("dress c0", "dress fock c"), ("dress c1", "dress fock a"), ("dress a2",),
                                       ("dress a3",))):
                for m in names:
                    chain[q].append((k, plan(by[m])))
            J = Operand.strided(e.G, {"P": n ** 3, "Q": n})
            K = Operand.strided(e.G, {"P": n ** 3, "Q": 1})
            last.append((nv(e.Fd, "PQ"), "PQ", [n] * 2, [term(J, "PQ", 2.0, o, n * n + 1),
                                                         term(K, "PQ", -1.0, o, n * n + n)], {"beta": 1.0}))
        upload_tables([g for c in chain for _, g in c])
        steps = [Combine(first)]
        for c in chain:
            steps += self._contractions(c)
        return steps + [Combine(last)]

    def _plan_update(self):
        """T3 -> r1, r2, W (TriplesEngine._setup_lower), denominators, norms and the T1/T2 update
        (rccsdt.py:916-931); the partials of the T3 terms of W stay for the intermediates."""
        operands, diag, build, gemms, final, dots = [], [], [], [], [], []
        for k, e in enumerate(self.engines):
            tr, o, v, n = e.tr, e.nocc, e.nvir, e.nmo
            lo = tr._lower
            nv = lambda b, l: Operand(b, l, b.shape)
            gv = lambda l: e.gview(e.G, l)
            ext = e.ext
            job = lambda b, l, ts, **opt: (nv(b, l), l, list(b.shape), ts, opt)
            oovv = gv("jkbc")
            operands += [job(lo["Ecomb"], "lija", [term(gv("ijla"), "lija", -1.0)]),          # [l,r,p,a]
                         job(lo["Evovv"], "cida", [term(gv("ciad"), "cida")]),
                         job(lo["Eoovv"], "jkbc", [term(oovv, "jkbc")]),
                         job(lo["Eoovv_t"], "jkcb", [term(oovv, "jkcb")]),
                         (Operand(lo["Er1"], "jkbcX", lo["Er1"].shape), "jkbc", [o, o, v, v],
                          [term(oovv, "jkbc"), term(gv("jkcb"), "jkbc", -0.5)], {})]
            diag.append((Operand.strided(lo["Ecomb"], {"l": o * o * v + o * v, "p": v, "a": 1}), "lpa", [o, o, v],
                         [term(Operand.strided(e.Fd, {"l": 0, "p": n, "a": 1}, o), "lpa", 0.5)], {"beta": 1.0}))
            build.append(Step(lambda _s, tr=tr: self._build_z(tr)))
            _, _, a2, a3 = lo["chunks"][0]
            ein = {g.name.split(" q0")[0]: g for g in a2 + a3 if isinstance(g, GemmLaunch)}
            # the E_ooov term as a partial of its own, after the o slices of the E_vovv term
            P2b = DeviceArray((o, o, v, v))
            Z = Operand(lo["Z"], "Qprabc", (o, o, o, v, v, v))
            zext = dict(ext, Q=o, r=o, p=o, l=o)
            ooov = plan_einsum("t3->r2 E_ooov", "Qprabc,lrpa->Qlbc", Z, Operand(lo["Ecomb"], "lrpa", (o, o, o, v)),
                               Operand(P2b, "Qlbc", (o, o, v, v)), 1.0, 0.0, zext, [({}, {}, {})])
            wvvvo = plan_einsum("t3->W_vvvo", "Qpreba,rpde->Qabd", Operand(lo["Z"], "Qpreba", (o, o, o, v, v, v)),
                                Operand(lo["Eoovv"], "rpde", (o, o, v, v)),
                                Operand(lo["dWovvv"], "Qabd", (o, v, v, v)), -1.0, 0.0, zext, [({}, {}, {})])
            for g in (ein["t3->r2 E_vovv"], ooov, ein["t3->r1"], ein["t3->W_vooo"], wvvvo):
                gemms.append((k, g))
            vv = v * v
            r2 = lambda l: Operand(e.r2, l, (o, o, v, v))
            p2 = lambda l: Operand(lo["P2"], l, (o, o, v, v))
            pb = lambda l: Operand(P2b, l, (o, o, v, v))
            self.arenas.append(P2b)
            final += [(nv(e.r1, "ia"), "ia", [o, v], [term(Operand(lo["P1"], "ia", (o, v)), "ia", 1.0, o * o, o * v)],
                       {"beta": 1.0, "acc": e.t1, "eia": e.eia, "rank": 1}),
                      (nv(e.r2s, "ijab"), "ijab", [o, o, v, v],
                       [t for l in ("ijab", "jiba") for t in (term(r2(l), "ijab"),
                                                              term(p2(l), "ijab", 1.0, o, o * o * vv),
                                                              term(pb(l), "ijab"))],
                       {"acc": e.t2, "eia": e.eia, "rank": 2})]
            dots += [(e.r1, e.r1, None, e.scal.ptr, e.r1.size, 0, 0),
                     (e.r2s, e.r2s, None, e.scal.ptr + 8, e.r2s.size, 0, 0)]
        upload_tables([g for _, g in gemms])
        return ([Combine(operands), Combine(diag)] + build + self._contractions(gemms) + [Combine(final), Dots(dots)])

    @staticmethod
    def _build_z(tr):
        """Z of the current T3.  The launches that follow reuse the buffer of the W_vvvo terms, so terms kept there
        by an earlier t3_to_r1r2 are no longer those of t3_to_w(reuse_z=True)."""
        tr._lower["dw_valid"] = False
        tr._build_z(0)

    def energies(self):
        """The energy dot products of every engine as one launch (into scal[2:4])."""
        jobs = []
        for e in self.engines:
            o, v = e.nocc, e.nvir
            jobs += [(e.Loovv, e.t2, e.t1, e.scal.ptr + 16, (o * v) ** 2, o, v),
                     (e.fov0, e.t1, None, e.scal.ptr + 24, o * v, 0, 0)]
        return Dots(jobs)

    def run(self, name, stream):
        for step in self.phases[name]:
            step.run(stream)
