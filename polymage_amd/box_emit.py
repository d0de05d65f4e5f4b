"""HIP emission of box kernels (see box_plan): group kernels whose tiles have
constant shapes.

The kernel has the two entry points and the tile decoding of every group
kernel (``hip_emit.wrap_kernel``); its body is two versions of the same
sweeps behind one workgroup-uniform test:

* inner tiles: every box lies inside its domain, its main Case and the
  arrays it reads.  No range check at all; global reads take a scalar base
  per (row, array) and one 32-bit byte offset per item;
* edge tiles: global reads clamp their coordinates, Cases are tested per
  point, stores to the output are tested against its domain, and blocks
  wholly outside a stage's domain are skipped.

Rows of LDS that a block reads at compile-time offsets are loaded in aligned
chunks of 4 or 2 elements: the row pitch and the block's stride are
multiples of the chunk, so its alignment is known at compile time.
"""

from .analysis import PlanError
from .box_plan import Known, Span, arg_map, const_int, fold, least_values
from .cprint import Printer, c_type
from .region_ir import bound_c

# device helpers of box kernels: a pointer moved by a byte offset, and
# stores of short vectors at element alignment (gfx950's global memory takes
# them unaligned).  The overloads keep the address space of the batch
# kernels' pointers.
BOX_PRELUDE = r'''
template <typename T, int N> struct pmx_vec {
  typedef T type __attribute__((vector_size(sizeof(T) * N)));
  typedef T utype __attribute__((vector_size(sizeof(T) * N), aligned(sizeof(T))));
};
#define PMX_STORES(AS) \
  template <typename T, int N> __device__ __forceinline__ void pmx_stv(T AS* p, typename pmx_vec<T, N>::type v) { \
    typedef typename pmx_vec<T, N>::utype U; *(U AS*)p = (U)v; } \
  template <typename T, int N> __device__ __forceinline__ void pmx_stv_nt(T AS* p, typename pmx_vec<T, N>::type v) { \
    typedef typename pmx_vec<T, N>::utype U; __builtin_nontemporal_store((U)v, (U AS*)p); } \
  template <typename T> __device__ __forceinline__ T AS* pmx_at(T AS* p, unsigned o) { return (T AS*)((char AS*)p + o); }
#define PMX_LOADS(AS) \
  template <typename T> __device__ __forceinline__ const T AS* pmx_at(const T AS* p, unsigned o) { return (const T AS*)((const char AS*)p + o); }
#define PMX_PLAIN
PMX_STORES(PMX_PLAIN)
PMX_LOADS(PMX_PLAIN)
#ifdef PMX_DEVICE_AS
PMX_STORES(PMX_GLOBAL)
PMX_LOADS(PMX_CONST)
#endif
'''


def _c(x):
    return str(x) if x >= 0 else '(%d)' % x


class _Body(object):
    """One version (inner or edge) of a box kernel's sweeps."""

    def __init__(self, plan, mode, threads, params, edge):
        self.plan = plan
        self.mode = mode
        self.threads = threads
        self.edge = edge
        self.base_pr = Printer({}, None, mode)
        self.L = []             # lines
        self.uni = {}           # uniform (scalar) pointers: key -> name
        self.uni_lines = []
        self.conds = {}         # inner tiles' conditions
        self.tmp = [0]
        self.final = set(plan.pipe.outputs) if plan.opts.get('nt_stores', 1) else set()

    # -- conditions of an inner tile ----------------------------------------------
    def need_ge(self, sp, lo, bound):
        """Inner tiles: coordinate ``sp.A * t + lo`` >= bound text."""
        k = ('>=', sp.d, sp.A, bound)
        self.conds[k] = min(lo, self.conds.get(k, lo))

    def need_le(self, sp, hi, bound):
        k = ('<=', sp.d, sp.A, bound)
        self.conds[k] = max(hi, self.conds.get(k, hi))

    def need_span(self, sp, lo_b, hi_b):
        self.need_ge(sp, sp.lo, lo_b)
        self.need_le(sp, sp.hi, hi_b)

    def need_apart(self, s, part):
        """Inner tiles: s's box does not meet the part's box."""
        terms = []
        for sp, (lo, hi) in zip(s.span, part.box):
            if lo is not None:
                terms.append('%s < %s' % (self.coord(sp, sp.hi), self.bound(lo)))
            if hi is not None:
                terms.append('%s > %s' % (self.coord(sp, sp.lo), self.bound(hi)))
        if not terms:
            raise PlanError("overlapping Cases")
        self.conds[('or', ' || '.join(terms))] = 0

    def bound(self, e):
        return '(%s)' % bound_c(e, self.base_pr)

    @staticmethod
    def coord(sp, c):
        if not sp.A:
            return _c(c)
        return '(t%d * %d + %s)' % (sp.d, sp.A, _c(c))

    def cond_lines(self):
        out = []
        for k in sorted(self.conds, key=str):
            if k[0] == 'or':
                out.append('(%s)' % k[1])
                continue
            op, d, A, b = k
            out.append('%s %s %s' % (self.coord(Span(d, A, 0, 0), self.conds[k]), op, b))
        return out

    # -- one point -----------------------------------------------------------------
    def known(self, s, u):
        value, mod = {}, {}
        for i, v in enumerate(s.func.variables):
            sp = s.span[i]
            if sp.A == 0 and s.cnt[i] == 1:
                value[v] = s.base[i] + u[i]
                continue
            m = sp.A
            if s.cnt[i] > 1:
                a, b = abs(m), s.blk[i]
                while b:
                    a, b = b, a % b
                m = a
            if m > 1:
                mod[v] = (m, (s.base[i] + u[i]) % m)
        return Known(value, mod)

    def parts_at(self, t, kn):
        """Parts of t that can apply at a point of known constants: those
        whose constant bounds admit its known coordinates."""
        out = []
        for part in t.parts:
            ok = True
            for v, (lo, hi) in zip(t.func.variables, part.box):
                x = kn.value.get(v)
                if x is None:
                    continue
                l, h = const_int(lo), const_int(hi)
                ok = ok and (l is None or x >= l) and (h is None or x <= h)
            if ok:
                out.append(part)
        return out

    def main_part(self, t, parts):
        """The part that covers most of t's domain at the estimates."""
        from .analysis import eval_bexpr
        dom = self.plan.pipe.domain_box(t.func)

        def vol(part):
            n = 1
            for (dlo, dhi), (lo, hi) in zip(dom, part.box):
                l = dlo if lo is None else max(dlo, eval_bexpr(lo, self.plan.env))
                h = dhi if hi is None else min(dhi, eval_bexpr(hi, self.plan.env))
                n *= max(0, h - l + 1)
            return n
        return max(parts, key=vol)


class _Item(object):
    """Addressing of one block of a sweep: stage ``s``, block indices
    ``j<i>``; ``u`` is the current point's offset in the block."""

    def __init__(self, body, s):
        self.B = body
        self.s = s
        self.u = [0] * s.nd
        self.decls = []
        self.names = {}
        self.probe = None       # LDS elements read: base -> set of offsets
        self.chunks = {}        # (base, first offset) -> (register, width)
        # edge tiles: the block's fixed-offset global reads, issued together
        # before its points: key -> (register, type, fast text, clamped text)
        self.early = {}
        # per array and kind of access: the block's first and last element;
        # and the ranges in which clamped indices do not clamp
        self.corner = {}
        self.free = {}

    def base(self, key, make):
        if key not in self.names:
            nm = 'ib%d' % len(self.names)
            self.names[key] = nm
            self.decls.append(make(nm))
        return self.names[key]

    def split(self, m, span_lo):
        """(constant, {block dim: stride}) of a map at the current point
        relative to the coordinate ``slope * A * t + span_lo``; None when the
        map is no fixed offset of the block."""
        s = self.s
        k = m.dim
        st = m.slope * s.blk[k]
        if s.cnt[k] > 1 and (s.blk[k] % m.period or st.denominator != 1):
            return None
        c = m.f(s.base[k] + self.u[k]) - span_lo
        return c, ({k: int(st)} if s.cnt[k] > 1 and st else {})

    def lds(self, p, ref, t, pr, pro):
        """Text of an LDS read of producer p."""
        W = [1] * p.nd
        for i in range(p.nd - 2, -1, -1):
            W[i] = W[i + 1] * p.lext[i + 1]
        const, coef, dyn = 0, {}, []
        for i, arg in enumerate(ref.arguments):
            m = arg_map(arg, t.func.variables)
            sp = p.lspan[i]
            if m.kind == 'const':
                const += (m.value - sp.lo) * W[i]
                continue
            if m.kind == 'var' and not (m.lows or m.highs):
                x = self.split(m, sp.lo)
                if x is not None:
                    const += x[0] * W[i]
                    for k, st in x[1].items():
                        coef[k] = coef.get(k, 0) + st * W[i]
                    continue
                q = pr.expr(arg, pro)
                dyn.append('__mul24(%s - %s, %d)' % (q, self.B.coord(sp, sp.lo), W[i]))
                continue
            q = pr.expr(arg, pro)
            if sp.A:
                # (a choice between two indices that are each as above: a
                # data-dependent index has no constant box but a constant
                # axis)
                dyn.append('__mul24(%s - %s, %d)' % (q, self.B.coord(sp, sp.lo), W[i]))
                continue
            q = 'pmx_clampi(%s, %d, %d)' % (q, p.span[i].lo, p.span[i].hi)
            dyn.append('__mul24(%s - %s, %d)' % (q, _c(sp.lo), W[i]))
        key = ('l', tuple(sorted(coef.items())))
        nm = self.base(key, lambda n: 'const int %s = %s;' % (n, ' + '.join(
            'j%d * %d' % kv for kv in sorted(coef.items())) or '0'))
        if dyn:
            return 'L_%s[%s + %d + %s]' % (p.name, nm, const, ' + '.join(dyn))
        if self.probe is not None:
            self.probe.setdefault((p.name, nm), (p, coef, set()))[2].add(const)
        for w in (16, 8, 4, 2):
            hit = self.chunks.get((p.name, nm, const // w * w, w))
            if hit:
                return '%s[%d]' % (hit, const % w)
        return 'L_%s[%s + %d]' % (p.name, nm, const)

    def gmem(self, f, ref, t, pr, pro, index_t='int'):
        """Text of a global read."""
        B = self.B
        maps = [arg_map(a, t.func.variables) for a in ref.arguments]
        nd = len(maps)
        # (edge tiles clamp every index of a data-dependent read: its other
        # indices may lie outside the array for points that do not count)
        static = not B.edge or all(m.kind != '*' for m in maps)
        xs = []
        dyn = []
        if static:
            for i, m in enumerate(maps):
                if m.kind == '*':
                    # clamped; its offset is added to the item's
                    q = 'pmx_clampi(%s, LB_%s_%d, LB_%s_%d + (int)E_%s_%d - 1)' % (
                        pr.expr(ref.arguments[i], pro), f.name, i, f.name, i, f.name, i)
                    dyn.append('(unsigned)(%s - LB_%s_%d) * %s' % (
                        q, f.name, i, '(unsigned)(S_%s_%d * %d)' % (f.name, i, f.typ.nbytes())
                        if i < nd - 1 else '%du' % f.typ.nbytes()))
                    xs.append(None)
                    continue
                if m.kind == 'const':
                    xs.append((m.value, {}, Span(None, 0, m.value, m.value)))
                    continue
                x = self.split(m, 0)
                sp = self.s.pspan[m.dim]
                if x is None or (m.slope * sp.A).denominator != 1 or (sp.A and sp.A % m.period):
                    static = False
                    break
                xs.append((x[0], x[1], Span(sp.d, int(m.slope * sp.A), m.f(sp.lo), m.f(sp.hi))))
        if static and not B.edge:
            for i, (m, x) in enumerate(zip(maps, xs)):
                if x is None:
                    continue
                B.need_span(x[2], B.bound(f.domain[i].lowerBound), B.bound(f.domain[i].upperBound))
                for b in m.lows:
                    B.need_ge(x[2], x[2].lo, B.bound(b))
                for b in m.highs:
                    B.need_le(x[2], x[2].hi, B.bound(b))
        if static:
            # scalar base of the row: every constant but the innermost's
            key = (f.name, tuple((x[2].d, x[2].A, x[0] if i < nd - 1 else 0) if x is not None else None
                                 for i, x in enumerate(xs)))
            if key not in B.uni:
                nm = 'gp%d' % len(B.uni)
                terms = []
                for i, k in enumerate(key[1]):
                    if k is None:
                        continue
                    d, A, c = k
                    e = '(%s)' % B.coord(Span(d, A, 0, 0), c)
                    terms.append('(%s - LB_%s_%d)%s' % (e, f.name, i, ' * S_%s_%d' % (f.name, i) if i < nd - 1 else ''))
                B.uni[key] = nm
                B.uni_lines.append('const auto %s = G_%s + (%s);' % (nm, f.name, ' + '.join(terms) or '0'))
            coef = {}
            for i, x in enumerate(xs):
                for k, st in (x[1] if x is not None else {}).items():
                    coef.setdefault(k, []).append((st, 'S_%s_%d' % (f.name, i) if i < nd - 1 else None))
            okey = ('g', f.typ.nbytes(), tuple(sorted((k, tuple(v)) for k, v in coef.items())))

            def mk(n):
                terms = []
                for k, v in sorted(coef.items()):
                    for st, S in v:
                        terms.append('(unsigned)j%d * %s' % (k, '(unsigned)(%s * %d)' % (S, st) if S else '%du' % st))
                return 'const unsigned %s = (%s) * %du;' % (n, ' + '.join(terms) or '0u', f.typ.nbytes())
            off = self.base(okey, mk)
            c = xs[-1][0] if nd and xs[-1] is not None else 0
            fast = 'pmx_at(%s, %s)[%d]' % (B.uni[key], ' + '.join([off] + dyn), c)
            if not B.edge:
                return fast
            # (reads of one element that are clamped differently differ in
            # their clamped form)
            ekey = (key, okey, c, tuple((tuple(B.bound(b) for b in m.lows), tuple(B.bound(b) for b in m.highs))
                                        for m in maps))
            if ekey not in self.early:
                reg = 'ge%d' % len(self.early)
                self.early[ekey] = (reg, c_type(f.typ), fast, self.clamped(f, ref, t))
            # corners of what the block reads of f, and where no clamp acts
            g = (f, tuple((tuple(sorted(x[1].items())), x[2].d, x[2].A) for x in xs))
            lo, hi = self.corner.get(g, ([x[0] for x in xs], [x[0] for x in xs]))
            self.corner[g] = ([min(v, x[0]) for v, x in zip(lo, xs)], [max(v, x[0]) for v, x in zip(hi, xs)])
            for i, (m, x) in enumerate(zip(maps, xs)):
                for b, op in [(b, '>=') for b in m.lows] + [(b, '<=') for b in m.highs]:
                    k = (op, B.bound(b), x[2].d, x[2].A, tuple(sorted(x[1].items())))
                    self.free[k] = (min if op == '>=' else max)(x[0], self.free.get(k, x[0]))
                if m.lows or m.highs:
                    for op, b in (('>=', f.domain[i].lowerBound), ('<=', f.domain[i].upperBound)):
                        k = (op, B.bound(b), x[2].d, x[2].A, tuple(sorted(x[1].items())))
                        self.free[k] = (min if op == '>=' else max)(x[0], self.free.get(k, x[0]))
            return self.early[ekey][0]
        e = None
        for i, arg in enumerate(ref.arguments):
            m = maps[i]
            q = pr.expr(arg, pro)
            if B.edge or m.kind == '*' or m.kind == 'var':
                q = 'pmx_clampi(%s, LB_%s_%d, LB_%s_%d + (int)E_%s_%d - 1)' % (
                    q, f.name, i, f.name, i, f.name, i)
            term = '(%s - LB_%s_%d)' % (q, f.name, i)
            e = term if e is None else '(%s * E_%s_%d + %s)' % (e, f.name, i, term)
        return 'G_%s[%s]' % (f.name, e or '0')

    def clamped(self, f, ref, t):
        """Text of a global read with every index clamped to the array, at
        the current point (coordinates from the item's base)."""
        names = self.coords(inline=True)
        pr = Printer(dict(zip(t.func.variables, names)), None, self.B.mode)
        e = None
        for i, arg in enumerate(ref.arguments):
            q = 'pmx_clampi(%s, LB_%s_%d, LB_%s_%d + (int)E_%s_%d - 1)' % (
                pr.expr(arg), f.name, i, f.name, i, f.name, i)
            term = '(%s - LB_%s_%d)' % (q, f.name, i)
            e = term if e is None else '(%s * E_%s_%d + %s)' % (e, f.name, i, term)
        return 'G_%s[%s]' % (f.name, e or '0')

    def safe(self):
        """C condition: every early read of the block, unclamped, stays inside
        its array (a read past a row's end lands in the neighbouring row: it
        serves no point that counts) and no index clamp acts."""
        out = []
        B = self.B
        for (f, kinds), corners in self.corner.items():
            nd = len(f.domain)
            total = ' * '.join('(long long)E_%s_%d' % (f.name, i) for i in range(nd))
            for which, cs in enumerate(corners):
                e = None
                for i, ((coef, d, A), c) in enumerate(zip(kinds, cs)):
                    q = '(%s%s - LB_%s_%d)' % (B.coord(Span(d, A, 0, 0), c), ''.join(
                        ' + j%d * %d' % kv for kv in coef), f.name, i)
                    e = '(long long)%s' % q if e is None else '(%s * E_%s_%d + %s)' % (e, f.name, i, q)
                out.append('%s < %s' % (e, total) if which else '%s >= 0' % e)
            if f.typ.nbytes() > 2:
                out.append('%s <= %dLL' % (total, 0xffffffff // f.typ.nbytes()))
        for (op, b, d, A, coef), c in sorted(self.free.items(), key=str):
            out.append('%s%s %s %s' % (B.coord(Span(d, A, 0, 0), c), ''.join(' + j%d * %d' % kv for kv in coef), op, b))
        return ' && '.join(out) or 'true'

    def ref_cb(self, t):
        plan = self.B.plan

        def cb(ref, pr, pro):
            f = ref.objectRef
            if plan.in_group(f):
                p = plan.stage_of(f)
                if p.inline:
                    return 'v_' + p.name
                return self.lds(p, ref, t, pr, pro)
            return self.gmem(f, ref, t, pr, pro)
        return cb

    # -- values --------------------------------------------------------------------
    def coords(self, inline=False):
        """(names, declarations) of the point's coordinates; ``inline``: the
        coordinates as expressions of the item's base."""
        if inline:
            return [_c(self.s.base[i] + self.u[i]) if sp.A == 0 and self.s.cnt[i] == 1 else
                    '(b%d + %d)' % (i, self.u[i]) for i, sp in enumerate(self.s.span)]
        names, decl = [], []
        for i, sp in enumerate(self.s.span):
            if sp.A == 0 and self.s.cnt[i] == 1:
                names.append(_c(self.s.base[i] + self.u[i]))
            else:
                names.append('q%d' % i)
                decl.append('const int q%d = b%d + %d;' % (i, i, self.u[i]))
        return names, decl

    def value(self, out, t, target, names, ind, flag):
        """Statements assigning stage t's value at the current point."""
        B = self.B
        plan = B.plan
        kn = B.known(self.s, self.u)
        # t's variables are s's, dimension by dimension (t is s or inlined)
        ren = dict(zip(self.s.func.variables, t.func.variables))
        kt = Known(dict((ren[v], x) for v, x in kn.value.items()),
                   dict((ren[v], x) for v, x in kn.mod.items()))
        parts = B.parts_at(t, kt)
        pr = Printer(dict(zip(t.func.variables, names)), self.ref_cb(t), B.mode, lazy=True,
                     exact_fma=not plan.opts.get('no_exact_fma'),
                     unify=None if plan.opts.get('no_unify') else (lambda r: self.cheap(t, r)))
        pr._tmp = B.tmp
        w = lambda x, i=ind: out.append('  ' * i + x)

        def assign(part, i):
            pro = []
            kp = Known(kt.value, kt.mod, least_values(t.func, part))
            val = pr.expr(fold(part.expr, kp), pro)
            for l in pro:
                w(l, i)
            w('%s = %s;%s' % (target, val, ' pmx_w = true;' if flag else ''), i)
        if not B.edge:
            if not parts:
                if t.liveout:
                    raise PlanError("an output point that no Case covers")
                return
            main = B.main_part(t, parts)
            const_cut = False
            for v, sp, (lo, hi) in zip(t.func.variables, t.span, main.box):
                l, h = const_int(lo), const_int(hi)
                if sp.A == 0 and v not in kt.value:
                    const_cut = const_cut or (l is not None and l > sp.lo) or (h is not None and h < sp.hi)
                if lo is not None and not (sp.A == 0 and l is not None):
                    B.need_ge(sp, sp.lo, B.bound(lo))
                if hi is not None and not (sp.A == 0 and h is not None):
                    B.need_le(sp, sp.hi, B.bound(hi))
            if const_cut:
                if t.liveout:
                    raise PlanError("a Case cuts a constant dimension of the output")
                # Cases that differ along a constant dimension the block
                # does not resolve: test per point, as at the edges
                self.tested(t, parts, names, assign, w, ind, kt)
                return
            for o in parts:
                if o is not main:
                    B.need_apart(t, o)
            assign(main, ind)
            return
        if len(parts) == 1 and not flag:
            assign(parts[0], ind)
            return
        self.tested(t, parts, names, assign, w, ind, kt)

    def tested(self, t, parts, names, assign, w, ind, kt):
        for part in parts:
            conds = []
            for v, nm, (lo, hi) in zip(t.func.variables, names, part.box):
                if v in kt.value:
                    x = kt.value[v]
                    if lo is not None and not (const_int(lo) is not None and const_int(lo) <= x):
                        conds.append('%s >= %s' % (nm, self.B.bound(lo)))
                    if hi is not None and not (const_int(hi) is not None and const_int(hi) >= x):
                        conds.append('%s <= %s' % (nm, self.B.bound(hi)))
                    continue
                if lo is not None:
                    conds.append('%s >= %s' % (nm, self.B.bound(lo)))
                if hi is not None:
                    conds.append('%s <= %s' % (nm, self.B.bound(hi)))
            if conds:
                w('if (%s) {' % ' && '.join(conds))
                assign(part, ind + 1)
                w('}')
            else:
                assign(part, ind)

    def cheap(self, t, r):
        f = r.objectRef
        if self.B.plan.in_group(f) and self.B.plan.stage_of(f).inline:
            return True
        for a in r.arguments:
            m = arg_map(a, t.func.variables)
            if m.kind == '*' or (m.kind == 'var' and self.split(m, 0) is None):
                return False
        return True

    def point(self, out, m, vname, wname, ind):
        """Value (and, at edges, coverage) of sweep member m at self.u."""
        B = self.B
        w = lambda x, i: out.append('  ' * i + x)
        names, decl = self.coords()
        w('{', ind)
        if decl:
            w(' '.join(decl), ind + 1)
        for t in self.inline_order(m):
            T = c_type(t.func.typ)
            w('%s v_%s = (%s)0;' % (T, t.name, T), ind + 1)
            w('{', ind + 1)
            self.value(out, t, 'v_' + t.name, names, ind + 2, False)
            w('}', ind + 1)
        if wname:
            w('bool pmx_w = false;', ind + 1)
        self.value(out, m, vname, names, ind + 1, bool(wname))
        if wname:
            w('%s = pmx_w;' % wname, ind + 1)
        w('}', ind)

    def inline_order(self, m):
        plan = self.B.plan
        out, seen = [], set()

        def visit(t):
            for part in t.parts:
                for r in plan._part_refs(part):
                    if plan.in_group(r.objectRef):
                        p = plan.stage_of(r.objectRef)
                        if p.inline and p not in seen:
                            seen.add(p)
                            visit(p)
                            out.append(p)
        visit(m)
        return out


def _sweep(B, members):
    """(comment, number of items, lines) of one sweep."""
    from .hip_emit import _magic24, _prod
    plan = B.plan
    s = members[0]
    nd = s.nd
    SL = []
    w = lambda x, ind=3: SL.append('  ' * ind + x)
    cnt = s.cnt
    nitems = _prod(cnt)
    rem = 'it'
    for i in range(nd):
        st = _prod(cnt[i + 1:])
        if cnt[i] == 1:
            w('const int j%d = 0; (void)j%d;' % (i, i))
        elif st == 1:
            w('const int j%d = %s;' % (i, rem))
        elif cnt[i] * st == nitems and nitems <= st:
            w('const int j%d = 0;' % i)
        else:
            mg = _magic24(cnt[i] * st, st)
            if st & (st - 1) == 0:
                sh = st.bit_length() - 1
                w('const int j%d = (int)((unsigned)%s >> %d); const int k%d = %s & %d;' % (
                    i, rem, sh, i, rem, st - 1))
            elif mg:
                w('const int j%d = (int)(__umul24((unsigned)%s, %du) >> %d); '
                  'const int k%d = %s - __mul24(j%d, %d);' % (i, rem, mg[0], mg[1], i, rem, i, st))
            else:
                w('const int j%d = %s / %d; const int k%d = %s - j%d * %d;' % (i, rem, st, i, rem, i, st))
            rem = 'k%d' % i
    for i, sp in enumerate(s.span):
        w('const int b%d = %s%s; (void)b%d;' % (i, B.coord(sp, s.base[i]),
                                               (' + j%d * %d' % (i, s.blk[i])) if cnt[i] > 1 else '', i))
    if B.edge:
        skip = []
        for i, sp in enumerate(s.span):
            if sp.A == 0:
                continue
            los = set(B.bound(m.func.domain[i].lowerBound) for m in members)
            his = set(B.bound(m.func.domain[i].upperBound) for m in members)
            if len(los) == 1 and len(his) == 1:
                skip.append('b%d > %s' % (i, his.pop()))
                skip.append('b%d + %d < %s' % (i, s.blk[i] - 1, los.pop()))
        if skip:
            w('if (%s) continue;' % ' || '.join(skip))
    import itertools
    pts = list(itertools.product(*[range(b) for b in s.blk]))
    item = _Item(B, s)

    def emit_points(out, flags):
        for mi, m in enumerate(members):
            for n, u in enumerate(pts):
                item.u = list(u)
                T = c_type(m.func.typ)
                out.append('  ' * 4 + '%s pv%d_%d = (%s)0;%s' % (
                    T, mi, n, T, ' bool pw%d_%d = false;' % (mi, n) if flags(m) else ''))
                item.point(out, m, 'pv%d_%d' % (mi, n), 'pw%d_%d' % (mi, n) if flags(m) else None, 4)

    flags = lambda m: B.edge and m.liveout
    # LDS rows read at fixed offsets, in aligned chunks
    item.probe = {}
    emit_points([], flags)
    loads = []
    vn = 0
    for (pname, nm), (p, coef, cs) in sorted(item.probe.items(), key=lambda kv: kv[0]):
        n = p.func.typ.nbytes()
        for w_ in (16, 8, 4, 2):
            if w_ * n > 16 or any(st % w_ for st in coef.values()):
                continue
            groups = {}
            for c in cs:
                groups.setdefault(c // w_ * w_, set()).add(c)
            size = p.lds_size // n
            hit = dict((g, v) for g, v in groups.items() if 2 * len(v) >= w_ and g + w_ <= size)
            if not hit:
                continue
            for g in sorted(hit):
                reg = 'lq%d' % vn
                vn += 1
                vt = 'pmx_vec<%s, %d>::type' % (c_type(p.func.typ), w_)
                loads.append('  ' * 4 + 'const %s %s = *(const %s*)(L_%s + (%s + %d));' % (vt, reg, vt, p.name, nm, g))
                item.chunks[(pname, nm, g, w_)] = reg
                cs -= hit[g]
    item.probe = None
    body = []
    emit_points(body, flags)
    for mi, m in enumerate(members):
        _stores(B, item, m, mi, pts, body)
    for d in item.decls:
        w(d)
    w('{')
    if item.early:
        # (clamping each read separately made the tiles at the image's edge,
        # a quarter of Harris' at 2048 x 2048, set the kernel's time)
        early = list(item.early.values())
        for reg, T, _, _ in early:
            w('%s %s;' % (T, reg), 4)
        w('if (%s) {' % item.safe(), 4)
        for reg, _, fast, _ in early:
            w('%s = %s;' % (reg, fast), 5)
        w('} else {', 4)
        for reg, _, _, slow in early:
            w('%s = %s;' % (reg, slow), 5)
        w('}', 4)
    SL.extend(loads)
    SL.extend(body)
    w('}')
    comment = 'stage %s (phase %d, %s points per thread)' % (
        ' + '.join(m.name for m in members), s.phase, 'x'.join(str(b) for b in s.blk) or '1')
    return comment, nitems, SL


def _runs(s, pts):
    """Points of a block grouped into runs along the innermost dimension."""
    rows = {}
    for n, u in enumerate(pts):
        rows.setdefault(u[:-1], []).append(n)
    return [rows[k] for k in sorted(rows)]


def _vec(T, names):
    return '(pmx_vec<%s, %d>::type){%s}' % (T, len(names), ', '.join(names))


def _pieces(names):
    """Runs of 4 or 2 names (vector stores) and single ones."""
    out, i = [], 0
    while i < len(names):
        n = 4 if len(names) - i >= 4 else (2 if len(names) - i >= 2 else 1)
        out.append((i, names[i:i + n]))
        i += n
    return out


def _stores(B, item, m, mi, pts, SL):
    w = lambda x, ind=4: SL.append('  ' * ind + x)
    s = item.s
    T = c_type(m.func.typ)
    if m.needs_lds:
        W = [1] * m.nd
        for i in range(m.nd - 2, -1, -1):
            W[i] = W[i + 1] * m.lext[i + 1]
        coef = {}
        for i in range(m.nd):
            if s.cnt[i] > 1:
                coef[i] = s.blk[i] * W[i]
        nm = item.base(('l', tuple(sorted(coef.items()))), lambda n: 'const int %s = %s;' % (
            n, ' + '.join('j%d * %d' % kv for kv in sorted(coef.items())) or '0'))
        for row in _runs(s, pts):
            c0 = sum((s.base[i] + pts[row[0]][i] - m.lspan[i].lo) * W[i] for i in range(m.nd))
            i = 0
            while i < len(row):
                n = 1
                for k in (4, 2):
                    if len(row) - i >= k and (c0 + i) % k == 0 and all(st % k == 0 for st in coef.values()):
                        n = k
                        break
                vals = ['pv%d_%d' % (mi, x) for x in row[i:i + n]]
                if n > 1:
                    vt = 'pmx_vec<%s, %d>::type' % (T, n)
                    w('*(%s*)(L_%s + (%s + %d)) = (%s){%s};' % (vt, m.name, nm, c0 + i, vt, ', '.join(vals)))
                else:
                    w('L_%s[%s + %d] = %s;' % (m.name, nm, c0 + i, vals[0]))
                i += n
    if not m.liveout:
        return
    f = m.func
    nt = f in B.final
    ptr = {}

    def at(u0):
        """Pointer to the output point at block offset u0 (a row's first)."""
        key = (f.name, 'st', tuple(u0[:-1]))
        if key not in B.uni:
            g = 'gp%d' % len(B.uni)
            terms = []
            for i in range(m.nd):
                c = s.base[i] + (u0[i] if i < m.nd - 1 else 0)
                terms.append('(%s - LB_%s_%d)%s' % (B.coord(s.span[i], c), f.name, i,
                                                    ' * S_%s_%d' % (f.name, i) if i < m.nd - 1 else ''))
            B.uni[key] = g
            e = ' + '.join(terms) or '0'
            B.uni_lines.append('const int %s = %s;' % (g, e) if B.edge else
                               'const auto %s = G_%s + (%s);' % (g, f.name, e))
        coef = tuple((i, s.blk[i]) for i in range(m.nd) if s.cnt[i] > 1)
        okey = ('gs', f.name)

        def mk(n):
            terms = []
            for i, b in coef:
                terms.append('(unsigned)j%d * %s' % (i, '(unsigned)(S_%s_%d * %d)' % (f.name, i, b)
                                                     if i < m.nd - 1 else '%du' % b))
            e = ' + '.join(terms) or '0u'
            return 'const unsigned %s = %s;' % (n, e if B.edge else '(%s) * %du' % (e, f.typ.nbytes()))
        # (the edge version serves every tile of an array above 4 GiB: its
        # offsets count elements, of which an array has fewer than 2^31)
        off = item.base(okey, mk)
        return '(G_%s + (%s + %s))' % (f.name, off, B.uni[key]) if B.edge else 'pmx_at(%s, %s)' % (B.uni[key], off)

    # points of a block that the box does not hold (its extent is no whole
    # number of blocks, or the block grid starts before it)
    def inside(u):
        c = []
        for i in range(m.nd):
            first = s.base[i] + u[i]
            last = first + (s.cnt[i] - 1) * s.blk[i]
            if first < s.span[i].lo:
                c.append('j%d > 0' % i if s.cnt[i] > 1 else 'false')
            if last > s.span[i].hi:
                c.append('j%d < %d' % (i, s.cnt[i] - 1) if s.cnt[i] > 1 else 'false')
        return c
    st = '__builtin_nontemporal_store(%s, &%s);' if nt else None

    def one(val, place):
        return (st % (val, place)) if nt else '%s = %s;' % (place, val)
    def vectors(p, row, ind):
        for i, vals in _pieces(['pv%d_%d' % (mi, n) for n in row]):
            c = pts[row[0]][-1] + i
            if len(vals) == 1:
                w(one(vals[0], '%s[%d]' % (p, c)), ind)
            else:
                w('pmx_stv%s<%s, %d>(%s + %d, %s);' % ('_nt' if nt else '', T, len(vals), p, c,
                                                      _vec(T, vals)), ind)
    if B.edge:
        for k, row in enumerate(_runs(s, pts)):
            p = at(list(pts[row[0]]))
            for n in row:
                u = pts[n]
                c = ['pw%d_%d' % (mi, n)] + inside(u)
                for i, sp in enumerate(s.span):
                    if sp.A:
                        c.append('b%d + %d >= %s' % (i, u[i], B.bound(f.domain[i].lowerBound)))
                        c.append('b%d + %d <= %s' % (i, u[i], B.bound(f.domain[i].upperBound)))
                w('const bool ok%d_%d = %s;' % (mi, n, ' && '.join(c)))
            if len(row) > 1:
                # whole runs as the inner tiles store them: separate stores
                # of neighbouring points leave lanes a stride apart
                w('if (%s) {' % ' && '.join('ok%d_%d' % (mi, n) for n in row))
                vectors(p, row, 5)
                w('} else {')
            for n in row:
                w('if (ok%d_%d) %s' % (mi, n, one('pv%d_%d' % (mi, n), '%s[%d]' % (p, pts[n][-1]))), 5)
            if len(row) > 1:
                w('}')
        return
    for i, sp in enumerate(s.span):
        if sp.A:
            B.need_span(sp, B.bound(f.domain[i].lowerBound), B.bound(f.domain[i].upperBound))
    for row in _runs(s, pts):
        p = at(list(pts[row[0]]))
        conds = [inside(pts[n]) for n in row]
        if all(c == conds[0] for c in conds):
            if conds[0]:
                w('if (%s) {' % ' && '.join(conds[0]))
            vectors(p, row, 5 if conds[0] else 4)
            if conds[0]:
                w('}')
            continue
        for n, c in zip(row, conds):
            x = one('pv%d_%d' % (mi, n), '%s[%d]' % (p, pts[n][-1]))
            w('if (%s) %s' % (' && '.join(c), x) if c else x)


def emit_box_kernel(pipe, plan, kname, threads, mode, xcd=True, forms=('plain', 'batch')):
    """(HIP source, KernelInfo) of one box kernel."""
    from .hip_emit import (KernelInfo, _prod, wrap_kernel, group_buffers, tile_lines, stride_lines, grid_exprs)
    params = pipe.sorted_parameters()
    reads, writes, buffers = group_buffers(plan)
    L = []
    w = lambda x, ind=1: L.append('  ' * ind + x)
    base_pr = Printer({}, None, mode)
    L.extend('  ' + l for l in tile_lines(plan, base_pr, xcd))
    L.extend('  ' + l for l in stride_lines(buffers, base_pr, 'int'))
    for s in plan.stages:
        if s.needs_lds:
            T = c_type(s.func.typ)
            w('%s* __restrict__ L_%s = (%s*)(pmx_lds + %d);' % (T, s.name, T, s.lds_offset))
    bodies = []
    for edge in (False, True):
        B = _Body(plan, mode, threads, params, edge)
        for s in plan.stages:
            if s.nd == 0:
                raise PlanError("a stage without dimensions")
        if not edge:
            # boxes inside their domains: nothing reads past a defined point
            for s in plan.stages:
                for i, sp in enumerate(s.span):
                    if sp.A:
                        B.need_span(sp, B.bound(s.func.domain[i].lowerBound),
                                    B.bound(s.func.domain[i].upperBound))
        first = True
        for ph in range(plan.nphases):
            sws = [_sweep(B, members) for (p, members) in plan.sweeps if p == ph]
            if not sws:
                continue
            if not first:
                B.L.append('  __syncthreads();')
            first = False
            B.L.append('  { // phase %d: %s' % (ph, '; '.join(c for (c, _, _) in sws)))
            # the sweeps of a phase one after another, each starting at the
            # wavefront after the last one's: no barrier between them, and
            # every wavefront runs one sweep's code at a time
            slots = [-(-n // 64) * 64 for (_, n, _) in sws]
            total = sum(slots[:-1]) + sws[-1][1]
            B.L.append('    for (int pmx_it = pmx_tx; pmx_it < %d; pmx_it += %d) {' % (total, threads))
            base = 0
            for k, (c, n, SL) in enumerate(sws):
                if len(sws) == 1:
                    B.L.append('    { const int it = pmx_it;')
                else:
                    B.L.append('    %sif (pmx_it < %d) { const int it = pmx_it - %d;' % (
                        '' if k == 0 else '} else ', base + slots[k] if k < len(sws) - 1 else total, base))
                    if n != slots[k] and k < len(sws) - 1:
                        B.L.append('      if (it >= %d) continue;' % n)
                B.L.extend(SL)
                base += slots[k]
            B.L.append('    }')
            B.L.append('    }')
            B.L.append('  }')
        bodies.append(B)
    inner, edge = bodies
    conds = inner.cond_lines()
    for f in buffers:
        if f.domain and f.typ.nbytes() > 2:
            # the inner tiles' byte offsets are 32-bit
            conds.append('%s <= %d' % (' * '.join('E_%s_%d' % (f.name, d) for d in range(len(f.domain))),
                                       0xffffffff // f.typ.nbytes()))
    w('if (%s) {' % (' && '.join(conds) or 'true'))
    L.extend('    ' + l for l in inner.uni_lines)
    L.extend(inner.L)
    w('} else {')
    L.extend('    ' + l for l in edge.uni_lines)
    L.extend(edge.L)
    w('}')
    grid_c, tiles_c = grid_exprs(plan, base_pr, 1)
    info = KernelInfo(kname, 'group', buffers, grid_c, threads, plan.lds_bytes, plan, reads, writes)
    info.tiles_c = tiles_c
    tiles = 1
    for n in plan.tile_space():
        tiles *= n
    info.work = tiles * sum(_prod([sp.ext for sp in s.span]) for s in plan.stages if not s.inline)
    return wrap_kernel(kname, params, buffers, writes, threads, plan.lds_bytes, L, forms), info
