"""Kernels for the groups that are not fused stencils.

* ``ConstPlan``: ``Function(..., "const")`` tables (look-up tables, colour
  matrices).  The reference never fuses them (grouping.py:146-161).  A
  table that depends only on parameters is computed on the host inside the
  stub with the host C library (the same libm the reference's g++ build
  uses, so ``powf``/``exp`` tables are bit-identical) and uploaded once per
  parameter change; a table that reads images is computed by a small
  per-point kernel.
* ``ReductionPlan``: ``Reduction`` stages (also never fused).  When every
  target index along a tiled dimension is a monotone floor-division map of
  one reduction variable (``2 + x/8``) the reduction is computed by
  "owner cells": each thread owns one cell of those dimensions, walks its
  pre-image of the reduction domain in the reference's lexicographic order
  and accumulates every data-dependent dimension (``2 + (int)(img*10)``) in
  LDS, or in registers when its cells have constant pre-images and few bins
  (``_emit_binned``), so the float sums are the reference's serial sums, bit for
  bit, with no atomics.  Reduction variables that appear in no target
  index (a row reduction ``hist(c, x) op= img(x, y)`` over y) are looped
  inside each owner thread in the domain's order, so those sums keep the
  reference's order too.  Integer reductions whose target is data
  dependent (histograms: ``hist(bin(img(x, y))) += 1``) have a result that
  does not depend on the order of their updates (integer +, *, min and max
  are associative and commutative, modulo 2^32 for + and *), so they run
  one thread per reduction point with device atomics, after a kernel that
  writes the default value.  The remaining cases (a float reduction into
  data-dependent cells with no owned dimension) run the reference's serial
  loop in a single thread (exact, slow).
"""

from fractions import Fraction

from .analysis import PlanError, always_refs, classify_access, case_parts, ceval_int, eval_bexpr, interval_image
from .constructs import Reference, Image, Case, Reduce, Op, Reduction, Parameter
from .cprint import Printer, c_type
from .expr_ast import Variable, Value
from .region_ir import bound_c


def _prod(xs):
    n = 1
    for x in xs:
        n *= x
    return n


def _extent_c(f, d, pr):
    return '(%s - %s + 1)' % (pr.expr(f.domain[d].upperBound), pr.expr(f.domain[d].lowerBound))


def _refs_of_parts(parts):
    refs = []
    for part in parts:
        refs += part.expr.collect(Reference)
        for c in part.pred:
            refs += c.collect(Reference)
    return refs


class ConstPlan(object):
    def __init__(self, pipe, group, gindex):
        self.pipe = pipe
        self.group = group
        self.gindex = gindex
        self.comp = group.comps[0]
        self.func = self.comp.func
        self.parts = self.comp.parts
        refs = _refs_of_parts(self.parts)
        self.on_host = len(refs) == 0
        self.params = pipe.sorted_parameters()
        self.upload_fn = 'pmx_upload_%s' % self.func.name

    def describe(self):
        return 'group %d: const table %s (%s)' % (self.gindex, self.func.name,
                                                  'host' if self.on_host else 'device')

    def host_code(self, pr, host_only=False):
        """C++ computing the table on the host (``<upload_fn>_host``) and,
        unless ``host_only``, uploading it to the device arena once per
        parameter key (``<upload_fn>``)."""
        f = self.func
        T = c_type(f.typ)
        nd = len(f.variables)
        names = ['h%d' % i for i in range(nd)]
        vn = dict(zip(f.variables, names))
        hp = Printer(vn, None, self.pipe.literal_mode)
        L = []
        w = L.append
        # host versions of the math helpers, once per translation unit
        w('#ifndef PMX_HOST_MATH')
        w('#define PMX_HOST_MATH')
        w('static inline float pmx_exp(float v) { return std::exp(v); }')
        w('static inline double pmx_exp(double v) { return std::exp(v); }')
        w('static inline double pmx_exp(int v) { return std::exp((double)v); }')
        w('static inline float pmx_sqrt(float v) { return std::sqrt(v); }')
        w('static inline double pmx_sqrt(double v) { return std::sqrt(v); }')
        w('static inline float pmx_abs(float v) { return std::abs(v); }')
        w('static inline double pmx_abs(double v) { return std::abs(v); }')
        w('static inline int pmx_abs(int v) { return std::abs(v); }')
        w('static inline float pmx_sin(float v) { return std::sin(v); }')
        w('static inline double pmx_sin(double v) { return std::sin(v); }')
        w('static inline float pmx_cos(float v) { return std::cos(v); }')
        w('static inline double pmx_cos(double v) { return std::cos(v); }')
        w('static inline double pmx_divc(double n, double r, double d) '
          '{ const double q = n * r; return std::fma(std::fma(-q, d, n), r, q); }')
        w('#endif')
        sig = ', '.join('%s %s' % (c_type(p.typ), p.name) for p in self.params)
        used = set(id(q) for q in f.getObjects(Parameter))
        keyp = [p for p in self.params if id(p) in used]
        w('static std::map<std::vector<unsigned char>, std::vector<%s> > pmx_tab_%s;' % (T, f.name))
        w('static std::set<std::pair<int, std::vector<unsigned char> > > pmx_tab_up_%s;' % f.name)
        # the host table (computed once per parameter key, kept for the
        # process) and its byte size
        w('static int %s_host(%s%sconst %s** data, size_t* bytes, std::vector<unsigned char>* keyp) {'
          % (self.upload_fn, sig, ', ' if sig else '', T))
        for p in self.params:
            w('  (void)%s;' % p.name)
        w('  std::vector<unsigned char> key;')
        for p in keyp:
            w('  { const unsigned char* q = (const unsigned char*)&%s; key.insert(key.end(), q, q + sizeof(%s)); }'
              % (p.name, p.name))
        size = ' * '.join('(long long)%s' % _extent_c(f, d, hp) for d in range(nd)) or '1'
        w('  long long n = %s;' % size)
        w('  std::vector<%s>& tab = pmx_tab_%s[key];' % (T, f.name))
        w('  if ((long long)tab.size() != n) {')
        w('    tab.assign((size_t)n, (%s)0);' % T)
        for i in range(nd):
            w('    ' + '  ' * i + 'for (int %s = %s; %s <= %s; ++%s) {' % (
                names[i], hp.expr(f.domain[i].lowerBound), names[i],
                hp.expr(f.domain[i].upperBound), names[i]))
        ind = '    ' + '  ' * nd
        lin = None
        for i in range(nd):
            t = '(long long)(%s - (%s))' % (names[i], hp.expr(f.domain[i].lowerBound))
            lin = t if lin is None else '(%s * %s + %s)' % (lin, _extent_c(f, i, hp), t)
        for part in self.parts:
            conds = []
            for i, (blo, bhi) in enumerate(part.box):
                if blo is not None:
                    conds.append('%s >= %s' % (names[i], bound_c(blo, hp)))
                if bhi is not None:
                    conds.append('%s <= %s' % (names[i], bound_c(bhi, hp)))
            pro = []
            pc = [hp.cond(c, pro) for c in part.pred]
            val = hp.expr(part.expr, pro)
            w(ind + 'if (%s) {' % (' && '.join(conds) or 'true'))
            for l in pro:
                w(ind + '  ' + l)
            w(ind + '  if (%s) tab[%s] = %s;' % (' && '.join(pc) or 'true', lin or '0', val))
            w(ind + '}')
        for i in reversed(range(nd)):
            w('    ' + '  ' * i + '}')
        w('  }')
        w('  *data = tab.data(); *bytes = (size_t)n * sizeof(%s);' % T)
        w('  if (keyp) *keyp = key;')
        w('  return 0;')
        w('}')
        if host_only:
            return L
        w('static int %s(%s%svoid* stream, void** out) {' % (self.upload_fn, sig, ', ' if sig else ''))
        w('  const %s* tdata = nullptr; size_t tbytes = 0; std::vector<unsigned char> key;' % T)
        w('  int rc = %s_host(%s%s&tdata, &tbytes, &key); if (rc) return rc;'
          % (self.upload_fn, ', '.join(p.name for p in self.params), ', ' if self.params else ''))
        w('  int dev = 0; if (hipGetDevice(&dev) != hipSuccess) return -1;')
        w('  unsigned long long h = 1469598103934665603ULL;')
        w('  for (unsigned char b : key) { h ^= b; h *= 1099511628211ULL; }')
        w('  char slot[128]; snprintf(slot, sizeof slot, "%s/const/%s/%%016llx", h);' % (self.pipe.name, f.name))
        w('  rc = pmx_arena_get(slot, tbytes, out); if (rc) return rc;')
        w('  if (!pmx_tab_up_%s.count(std::make_pair(dev, key))) {' % f.name)
        w('    rc = pmx_memcpy_h2d(*out, tdata, tbytes, stream); if (rc) return rc;')
        w('    rc = pmx_stream_sync(stream); if (rc) return rc;')
        w('    pmx_tab_up_%s.insert(std::make_pair(dev, key));' % f.name)
        w('  }')
        w('  return 0;')
        w('}')
        return L


def emit_const_kernel(pipe, plan, kname, mode):
    """One thread per table point; the table reads images (e.g. a colour
    matrix interpolated from two input matrices)."""
    from .hip_emit import KernelInfo, wrap_kernel
    f = plan.func
    params = pipe.sorted_parameters()
    reads = []
    for r in _refs_of_parts(plan.parts):
        if r.objectRef not in reads:
            reads.append(r.objectRef)
    buffers = sorted(reads, key=lambda g: g.name) + [f]
    nd = len(f.variables)
    names = ['p%d' % i for i in range(nd)]
    base = Printer({}, None, mode)

    def cb(ref, pr, pro):
        g = ref.objectRef
        lin = None
        for d, arg in enumerate(ref.arguments):
            q = 'pmx_clampi(%s, %s, %s)' % (pr.expr(arg, pro), base.expr(g.domain[d].lowerBound),
                                             base.expr(g.domain[d].upperBound))
            t = '(%s - (%s))' % (q, base.expr(g.domain[d].lowerBound))
            lin = t if lin is None else '(%s * %s + %s)' % (lin, _extent_c(g, d, base), t)
        return 'G_%s[%s]' % (g.name, lin or '0')
    pr = Printer(dict(zip(f.variables, names)), cb, mode, lazy=True)
    args = ['const %s %s' % (c_type(p.typ), p.name) for p in params]
    for g in buffers:
        if g is f:
            args.append('%s* __restrict__ G_%s' % (c_type(g.typ), g.name))
        else:
            args.append('const %s* __restrict__ G_%s' % (c_type(g.typ), g.name))
    L = []
    w = lambda s: L.append('  ' + s)
    exts = [_extent_c(f, d, base) for d in range(nd)]
    w('long long pmx_n = %s;' % (' * '.join('(long long)%s' % e for e in exts) or '1'))
    w('long long idx = (long long)pmx_tile * 256 + threadIdx.x;')
    w('if (idx >= pmx_n) return;')
    w('long long rem = idx;')
    for i in reversed(range(nd)):
        w('const int %s = (int)(rem %% %s) + (%s); rem /= %s;' % (
            names[i], exts[i], base.expr(f.domain[i].lowerBound), exts[i]))
    w('%s v = (%s)0; bool pmx_w = false;' % (c_type(f.typ), c_type(f.typ)))
    for part in plan.parts:
        conds = []
        for i, (blo, bhi) in enumerate(part.box):
            if blo is not None:
                conds.append('%s >= %s' % (names[i], bound_c(blo, base)))
            if bhi is not None:
                conds.append('%s <= %s' % (names[i], bound_c(bhi, base)))
        w('if (%s) {' % (' && '.join(conds) or 'true'))
        pro = []
        pc = [pr.cond(c, pro) for c in part.pred]
        val = pr.expr(part.expr, pro)
        for l in pro:
            w('  ' + l)
        w('  if (%s) { v = %s; pmx_w = true; }' % (' && '.join(pc) or 'true', val))
        w('}')
    w('if (pmx_w) G_%s[idx] = v;' % f.name)
    grid = '((%s + 255) / 256)' % (' * '.join('(long long)%s' % e for e in exts) or '1')
    info = KernelInfo(kname, 'const', buffers, grid, 256, 0, plan,
                      [g for g in buffers if g is not f], [f])
    return wrap_kernel(kname, params, buffers, [f], 256, 0, L), info


class _RedCase(object):
    def __init__(self, cond, red, index):
        self.cond = cond
        self.red = red
        self.index = index


class ReductionPlan(object):
    """See module docstring.  ``owner`` is True when the owner-cell kernel
    applies; ``owned`` maps each reduction variable to the target dimension
    it owns."""

    MAX_ACC = 64

    def __init__(self, pipe, group, gindex):
        self.pipe = pipe
        self.group = group
        self.gindex = gindex
        self.comp = group.comps[0]
        f = self.func = self.comp.func
        self.rvars = list(f.reductionVariables)
        self.fvars = list(f.variables)
        self.cases = []
        for i, case in enumerate(f.defn):
            if isinstance(case, Case):
                self.cases.append(_RedCase(case.condition, case.expression, i))
            else:
                self.cases.append(_RedCase(None, case, i))
        for rc in self.cases:
            if not isinstance(rc.red, Reduce):
                raise PlanError("reduction %s: definition must be Reduce" % f.name)
        self._classify()

    def _classify(self):
        f = self.func
        nd = len(self.fvars)
        owned = {}
        self.pre_size = {}
        ok = True
        self.loop_vars = []
        for j, rv in enumerate(self.rvars):
            dim = None
            hits = []
            for rc in self.cases:
                tgt = rc.red.accumulate_ref.arguments
                hit = [d for d in range(nd)
                       if classify_access(tgt[d], self.rvars).kind == 'var'
                       and classify_access(tgt[d], self.rvars).var is rv]
                hits.append(hit)
            if all(not h for h in hits) and not any(
                    rv in [v for v in _vars_of(rc.red.accumulate_ref.arguments[d])]
                    for rc in self.cases for d in range(nd)
                    if classify_access(rc.red.accumulate_ref.arguments[d], self.rvars).kind != '*'):
                # in no affine target index: every owner thread walks it
                self.loop_vars.append(rv)
                continue
            for rc, hit in zip(self.cases, hits):
                tgt = rc.red.accumulate_ref.arguments
                if len(hit) != 1:
                    ok = False
                    break
                if dim is None:
                    dim = (hit[0], str(tgt[hit[0]]))
                elif dim != (hit[0], str(tgt[hit[0]])):
                    ok = False
                    break
            if not ok or dim is None:
                ok = False
                break
            acc = classify_access(rc.red.accumulate_ref.arguments[dim[0]], self.rvars)
            if not acc.increasing:
                ok = False
                break
            owned[rv] = dim[0]
            # cells own k consecutive values of rv when the access is rv/k + c
            if acc.slope.numerator == 1 and acc.slope.denominator > 1:
                self.pre_size[rv] = int(acc.slope.denominator)
        env = self.pipe.param_env
        self.free_dims = [d for d in range(nd) if d not in owned.values()]
        nacc = 1
        for d in self.free_dims:
            lo = ceval_int(f.domain[d].lowerBound, env)
            hi = ceval_int(f.domain[d].upperBound, env)
            nacc *= (hi - lo + 1)
        self.nacc = nacc
        self.owner = ok and bool(owned) and len(owned) + len(self.loop_vars) == len(self.rvars) \
            and nacc <= self.MAX_ACC
        self.owned = owned
        self.bin_dim = self._bins() if self.owner and not self.pipe.gpu_options.get('no_bins') else None
        self.atomic = (not self.owner) and self._atomic_ok()

    # registers of a binned owner thread's accumulators
    MAX_BINS = 16

    def _bins(self):
        """The one data-dependent free dimension (constant extent) of an
        owner-cell reduction whose other free dimensions every case targets
        at constants and whose cells have constant pre-images: its cells'
        accumulators then fit in registers (_emit_binned).  None if there is
        no such dimension, or accumulators in LDS are faster."""
        f = self.func
        ks = [self.pre_size.get(rv) for rv in self.rvars]
        if not all(ks) or _prod_int(ks) > 256:
            return None
        data = set()
        for rc in self.cases:
            for d in self.free_dims:
                acc = classify_access(rc.red.accumulate_ref.arguments[d], self.rvars)
                if acc.kind == '*':
                    data.add(d)
                elif acc.kind != 'const':
                    return None
        if len(data) != 1:
            return None
        z = data.pop()
        try:
            consts = [[ceval_int(rc.red.accumulate_ref.arguments[d], {}) for d in self.free_dims if d != z]
                      for rc in self.cases
                      if classify_access(rc.red.accumulate_ref.arguments[z], self.rvars).kind == '*']
            ext = dict((d, ceval_int(f.domain[d].upperBound, {}) - ceval_int(f.domain[d].lowerBound, {}) + 1)
                       for d in self.free_dims)
        except (PlanError, KeyError):
            return None
        other = _prod_int([e for d, e in ext.items() if d != z])
        half = (ext[z] + 1) // 2
        if len(consts) != len(self.cases) or ext[z] < 2 or half * other > self.MAX_BINS:
            return None
        # Against LDS accumulators, times of LDS / registers at 300 x 400,
        # 1083 x 1923 and 2560 x 1536 (whose cells are all whole):
        # every bin costs a thread a compare and an update per point, more
        # than one LDS update beyond 8 bins: 32 bins on 8 x 8 cells 0.93 0.87
        # 0.58, 16 bins 1.44 1.21 0.79, 8 bins 2.01 1.55 1.00;
        # cells of few points have wavefronts enough to hide the LDS, unless
        # it holds many accumulators: 2 x 2 cells, 8 bins 0.98 0.94 0.93, 12
        # bins 0.99 1.20 1.23; 4 x 2 cells, 6 bins 0.96 1.02 0.81; 4 x 4, 8
        # bins 1.00 1.32 0.76; 8 x 4, 4 bins 1.93 2.18 0.91;
        # a Case decided at run time keeps its reads behind it, so that they
        # no longer issue together: 8 x 8 cells, two planes of 14 bins 0.54
        # 0.62 1.13, of 4 bins 0.58 0.60 1.03 - only small cells with more
        # accumulators than the LDS kernel holds well gain then: 4 x 4 cells,
        # two planes of 8 bins 0.96 0.75 0.75, of 10 bins 1.15 1.18 1.56.
        points, acc = _prod_int(ks), ext[z] * other
        if half > 8:
            return None
        if any(_decided(self, rc) is None for rc in self.cases):
            return z if points <= 16 and other > 1 and acc > 16 else None
        return z if points >= 8 or acc >= 12 else None

    def floor_start(self, rv, arg, lower):
        """f0 when ``arg`` is f0 + rv / k for every rv >= 0 the domain holds
        (k = pre_size), else None."""
        k = self.pre_size.get(rv)
        if k is None or any(type(v) is not Variable or v is not rv for v in arg.collect(Variable)):
            return None
        try:
            if ceval_int(lower, {}) < 0:
                return None
            f0 = ceval_int(arg, {rv: 0})
            same = all(ceval_int(arg, {rv: r}) == f0 + r // k for r in range(4 * k))
        except (PlanError, KeyError):
            return None
        return f0 if same else None

    def _atomic_ok(self):
        """Integer target, integer values of the target's promoted type and
        an operator whose result is independent of the update order."""
        from .expression import getType
        from .expr_types import Int, UInt, Char, UChar, Short, UShort
        f = self.func
        if f.typ not in (Int, UInt):
            return False
        for rc in self.cases:
            if rc.red.op_type not in (Op.Sum, Op.Mul, Op.Min, Op.Max):
                return False
            vt = getType(rc.red.expression)
            if vt in (Char, UChar, Short, UShort):
                vt = Int
            if vt is not f.typ:
                return False
        return True

    def describe(self):
        kind = 'owner cells' if self.owner else ('atomic' if self.atomic else 'serial')
        return 'group %d: reduction %s (%s, %d accumulators per cell)' % (
            self.gindex, self.func.name, kind, self.nacc)


def _vars_of(e):
    return e.collect(Variable) if hasattr(e, 'collect') else []


def _cond_dims(plan, rc):
    """Dimensions of the function's own variables in a case's condition."""
    if rc.cond is None:
        return []
    used = rc.cond.collect(Variable)
    return [d for d, v in enumerate(plan.fvars) if v not in plan.rvars and any(v is u for u in used)]


def _decided(plan, rc):
    """True, False or None (not known) for a case's condition when it is on
    nothing but the function's dimensions that the case targets at
    constants; True without a condition."""
    from .box_plan import Known, decide
    if rc.cond is None:
        return True
    value = {}
    for d in _cond_dims(plan, rc):
        try:
            value[plan.fvars[d]] = ceval_int(rc.red.accumulate_ref.arguments[d], {})
        except PlanError:
            return None
    try:
        return decide(rc.cond, Known(value, {}))
    except PlanError:
        return None


def _prod_int(xs):
    n = 1
    for x in xs:
        n *= x
    return n


def _reads_of_reduction(plan):
    reads = []
    for rc in plan.cases:
        refs = rc.red.expression.collect(Reference)
        refs += [r for r in rc.red.accumulate_ref.collect(Reference) if r is not rc.red.accumulate_ref]
        if rc.cond is not None:
            refs += rc.cond.collect(Reference)
        for r in refs:
            if r.objectRef is not plan.func and r.objectRef not in reads:
                reads.append(r.objectRef)
    return reads


def emit_reduction_kernel(pipe, plan, kname, mode):
    from .hip_emit import KernelInfo, wrap_kernel
    f = plan.func
    params = pipe.sorted_parameters()
    reads = _reads_of_reduction(plan)
    buffers = sorted(reads, key=lambda g: g.name) + [f]
    base = Printer({}, None, mode)
    T = c_type(f.typ)
    nd = len(plan.fvars)
    rnames = ['r%d' % j for j in range(len(plan.rvars))]

    def cb(ref, pr, pro):
        g = ref.objectRef
        lin = None
        for d, arg in enumerate(ref.arguments):
            q = pr.expr(arg, pro)
            acc = classify_access(arg, plan.rvars)
            if acc.kind == '*':
                q = 'pmx_clampi(%s, %s, %s)' % (q, base.expr(g.domain[d].lowerBound),
                                                base.expr(g.domain[d].upperBound))
            t = '(%s - (%s))' % (q, base.expr(g.domain[d].lowerBound))
            lin = t if lin is None else '(%s * %s + %s)' % (lin, _extent_c(g, d, base), t)
        return 'G_%s[%s]' % (g.name, lin or '0')

    args = ['const %s %s' % (c_type(p.typ), p.name) for p in params]
    for g in buffers:
        if g is f:
            args.append('%s* __restrict__ G_%s' % (T, g.name))
        else:
            args.append('const %s* __restrict__ G_%s' % (c_type(g.typ), g.name))
    L = []
    w = lambda s, ind=1: L.append('  ' * ind + s)
    exts = [_extent_c(f, d, base) for d in range(nd)]
    lbs = [base.expr(f.domain[d].lowerBound) for d in range(nd)]

    def red_body(ind, target_ok, update=None):
        """Statements processing the current reduction point (names
        r0..rk bound).  ``target_ok(dimvals)`` filters owned cells;
        ``update(op, val)`` gives the statement applying one value (by
        default the C update of ``acc_slot()``)."""
        pr = Printer(dict(zip(plan.rvars, rnames)), cb, mode, lazy=True)
        for rc in plan.cases:
            red = rc.red
            tgt = red.accumulate_ref.arguments
            w('{', ind)
            # a Case's condition guards the reads of its value and of its
            # target; only the coordinates it is on come before it
            first = _cond_dims(plan, rc)
            for d in first:
                target(pr, tgt, d, ind + 1)
            conds = []
            if rc.cond is not None:
                vn = dict(zip(plan.rvars, rnames))
                for v, d in zip(plan.fvars, range(nd)):
                    if v not in plan.rvars:
                        vn[v] = 'q%d' % d
                cpr = Printer(vn, cb, mode, lazy=True)
                cpro = []
                cc = cpr.cond(rc.cond, cpro)
                for l in cpro:
                    w(l, ind + 1)
                w('if (%s) {' % cc, ind + 1)
            for d in range(nd):
                if d not in first:
                    target(pr, tgt, d, ind + 1)
            pro = []
            val = pr.expr(red.expression, pro)
            for l in pro:
                w(l, ind + 1)
            extra = target_ok()
            if extra:
                conds.append(extra)
            op = red.op_type
            if update is not None:
                upd = update(op, val)
            else:
                slot = acc_slot()
                if op == Op.Sum:
                    upd = '%s = (%s + %s);' % (slot, slot, val)
                elif op == Op.Mul:
                    upd = '%s = (%s * %s);' % (slot, slot, val)
                elif op == Op.Min:
                    upd = '%s = ((%s < %s)? (%s)(%s): %s);' % (slot, val, slot, T, val, slot)
                else:
                    upd = '%s = ((%s > %s)? (%s)(%s): %s);' % (slot, val, slot, T, val, slot)
            w('if (%s) { %s }' % (' && '.join(conds) or 'true', upd), ind + 1)
            w('}' if rc.cond is None else '} }', ind)

    def target(pr, tgt, d, ind):
        """q<d>: the target's coordinate of dimension d."""
        pro = []
        q = pr.expr(tgt[d], pro)
        if classify_access(tgt[d], plan.rvars).kind == '*':
            q = 'pmx_clampi(%s, %s, %s)' % (q, lbs[d], base.expr(f.domain[d].upperBound))
        for l in pro + ['const int q%d = %s;' % (d, q)]:
            w(l, ind)

    def preimage():
        """lo<j>/hi<j>: the cell's points along every reduction variable."""
        # pre-image of the cell along every owned reduction variable; the
        # other reduction variables are walked over their whole range
        for j, rv in enumerate(plan.rvars):
            if rv not in plan.owned:
                w('const int lo%d = %s, hi%d = %s;' % (
                    j, base.expr(f.reductionDomain[j].lowerBound), j,
                    base.expr(f.reductionDomain[j].upperBound)))
                continue
            d = plan.owned[rv]
            arg = plan.cases[0].red.accumulate_ref.arguments[d]
            rlo = base.expr(f.reductionDomain[j].lowerBound)
            rhi = base.expr(f.reductionDomain[j].upperBound)
            f0 = plan.floor_start(rv, arg, f.reductionDomain[j].lowerBound)
            if f0 is not None:
                # f(r) = f0 + r / k: the cell's points in closed form (the
                # searches below are a chain of some 20 dependent steps)
                k = plan.pre_size[rv]
                w('const int lo%d = pmx_imax(%s, (c%d - (%d)) * %d), hi%d = pmx_imin(%s, (c%d - (%d)) * %d + %d);'
                  % (j, rlo, d, f0, k, j, rhi, d, f0, k, k - 1))
                continue
            fpr = Printer({rv: 'm'}, cb, mode, lazy=True)
            fx = fpr.expr(arg)
            # lo_j = first r with f(r) >= c ; hi_j = last r with f(r) <= c
            w('int lo%d, hi%d;' % (j, j))
            w('{ int a = %s, b = %s + 1;' % (rlo, rhi))
            w('  while (a < b) { const int m = a + (b - a) / 2; if ((%s) >= c%d) b = m; else a = m + 1; }' % (fx, d))
            w('  lo%d = a; }' % j)
            w('{ int a = %s - 1, b = %s;' % (rlo, rhi))
            w('  while (a < b) { const int m = a + (b - a + 1) / 2; if ((%s) <= c%d) a = m; else b = m - 1; }' % (fx, d))
            w('  hi%d = a; }' % j)

    if plan.owner and plan.bin_dim is not None:
        return _emit_binned(pipe, plan, kname, mode, params, reads, buffers, exts, lbs, base, cb, rnames,
                            preimage, L)

    if plan.owner:
        # thread per owned cell; accumulators for the free dims in LDS
        od = sorted(plan.owned.values())
        free = plan.free_dims
        nthreads = 256
        w('%s* pmx_acc = (%s*)pmx_lds;' % (T, T))
        w('%s* acc = pmx_acc + threadIdx.x;' % T)
        ncell = ' * '.join('(long long)%s' % exts[d] for d in od)
        w('const long long pmx_ncell = %s;' % ncell)
        w('long long cell = (long long)pmx_tile * %d + threadIdx.x;' % nthreads)
        w('if (cell >= pmx_ncell) return;')
        for d in reversed(od):
            w('const int c%d = (int)(cell %% %s) + (%s); cell /= %s;' % (d, exts[d], lbs[d], exts[d]))
        # free-dim strides in the accumulator array
        fext = [exts[d] for d in free]

        def acc_index(names):
            e = None
            for k, d in enumerate(free):
                t = '(%s - (%s))' % (names[d], lbs[d])
                e = t if e is None else '(%s * %s + %s)' % (e, fext[k], t)
            return '(%s) * %d' % (e or '0', nthreads)
        # init with the default value
        dvn = {}
        w('for (int a = 0; a < %d; ++a) {' % plan.nacc)
        rem = 'a'
        fn = {}
        for k in reversed(range(len(free))):
            d = free[k]
            w('  const int f%d = (%s) %% %s + (%s);' % (d, rem, fext[k], lbs[d]))
            w('  const int a%d = (%s) / %s;' % (d, rem, fext[k]))
            rem = 'a%d' % d
            fn[d] = 'f%d' % d
        names = dict((d, 'c%d' % d) for d in od)
        names.update(fn)
        dpr = Printer(dict((plan.fvars[d], names[d]) for d in range(nd)), cb, mode, lazy=True)
        w('  acc[a * %d] = %s;' % (nthreads, dpr.expr(f.default)))
        w('}')
        preimage()
        def acc_slot_owner():
            nm = dict((d, 'q%d' % d) for d in free)
            return 'acc[%s]' % acc_index(nm)
        acc_slot = acc_slot_owner

        def owned_ok():
            return ' && '.join('q%d == c%d' % (d, d) for d in od)

        ks = [plan.pre_size.get(rv) for rv in plan.rvars]
        fast = all(ks) and _prod_int(ks) <= 256
        if fast:
            # interior cells own a full k0 x k1 x ... pre-image: constant trip
            # counts, fully unrolled, so all its loads issue up front (the
            # order of the accumulations, hence every sum, is unchanged)
            w('if (%s) {' % ' && '.join('hi%d - lo%d + 1 == %d' % (j, j, k) for j, k in enumerate(ks)))
            ind = 2
            for j, k in enumerate(ks):
                w('#pragma unroll', ind)
                w('for (int i%d = 0; i%d < %d; ++i%d) { const int r%d = lo%d + i%d;' % (j, j, k, j, j, j, j), ind)
                ind += 1
            red_body(ind, lambda: '')
            for j in reversed(range(len(plan.rvars))):
                ind -= 1
                w('}', ind)
            w('} else {')
        ind = 2 if fast else 1
        for j in range(len(plan.rvars)):
            w('for (int r%d = lo%d; r%d <= hi%d; ++r%d) {' % (j, j, j, j, j), ind)
            ind += 1
        red_body(ind, owned_ok)
        for j in reversed(range(len(plan.rvars))):
            ind -= 1
            w('}', ind)
        if fast:
            w('}')
        # write out the cell's slice of the grid
        w('for (int a = 0; a < %d; ++a) {' % plan.nacc)
        rem = 'a'
        for k in reversed(range(len(free))):
            d = free[k]
            w('  const int f%d = (%s) %% %s + (%s);' % (d, rem, fext[k], lbs[d]))
            w('  const int a%d = (%s) / %s;' % (d, rem, fext[k]))
            rem = 'a%d' % d
        lin = None
        for d in range(nd):
            t = '(long long)(%s - (%s))' % (names[d], lbs[d])
            lin = t if lin is None else '(%s * %s + %s)' % (lin, exts[d], t)
        w('  G_%s[%s] = acc[a * %d];' % (f.name, lin, nthreads))
        w('}')
        grid = '((%s + %d) / %d)' % (ncell, nthreads - 1, nthreads)
        lds = nthreads * plan.nacc * f.typ.nbytes()
        info = KernelInfo(kname, 'reduction', buffers, grid, nthreads, lds, plan, reads, [f])
        return [(wrap_kernel(kname, params, buffers, [f], nthreads, lds, L), info)]

    if plan.atomic:
        return _emit_atomic(pipe, plan, kname, mode, params, reads, buffers, exts, lbs, base,
                            red_body, L)

    # serial fallback: one thread, the reference loop order
    w('if (threadIdx.x != 0) return;')
    lin = None
    ind = 1
    for d in range(nd):
        w('for (int f%d = %s; f%d <= %s; ++f%d) {' % (d, lbs[d], d, base.expr(f.domain[d].upperBound), d), ind)
        ind += 1
        t = '(long long)(f%d - (%s))' % (d, lbs[d])
        lin = t if lin is None else '(%s * %s + %s)' % (lin, exts[d], t)
    dpr = Printer(dict((plan.fvars[d], 'f%d' % d) for d in range(nd)), cb, mode, lazy=True)
    w('G_%s[%s] = %s;' % (f.name, lin or '0', dpr.expr(f.default)), ind)
    for d in reversed(range(nd)):
        ind -= 1
        w('}', ind)
    for j in range(len(plan.rvars)):
        w('for (int r%d = %s; r%d <= %s; ++r%d) {' % (
            j, base.expr(f.reductionDomain[j].lowerBound), j,
            base.expr(f.reductionDomain[j].upperBound), j), ind)
        ind += 1
    tl = None
    for d in range(nd):
        t = '(long long)(q%d - (%s))' % (d, lbs[d])
        tl = t if tl is None else '(%s * %s + %s)' % (tl, exts[d], t)

    def acc_slot():
        return 'G_%s[%s]' % (f.name, tl or '0')
    red_body(ind, lambda: None)
    for j in reversed(range(len(plan.rvars))):
        ind -= 1
        w('}', ind)
    info = KernelInfo(kname, 'reduction', buffers, '1', 64, 0, plan, reads, [f])
    return [(wrap_kernel(kname, params, buffers, [f], 64, 0, L), info)]


def _emit_binned(pipe, plan, kname, mode, params, reads, buffers, exts, lbs, base, cb, rnames, preimage, L):
    """Owner cells whose data-dependent dimension (``plan.bin_dim``) is held
    in registers, two threads per cell, each with half of the bins.

    A thread walks its cell's points in the domain's order and updates, of
    its bins, the one the value selects: a compare and a conditional update
    per bin, all of them independent, so the vector issue rate bounds it
    (33 instructions per pixel and thread).  The owner kernel with LDS
    accumulators waits, for every value, for a read, an addition and a
    write, and its few wavefronts (993 for the grid of a 2560 x 1536 image,
    on 1,024 SIMDs) hide none of it; LDS float atomics, which need no wait,
    were slower still (46 us).  Two threads a cell double the wavefronts at
    the price of reading the image twice (from L1), and workgroups of one
    wavefront spread them over all compute units.  Grid kernel of a
    2560 x 1536 image 16.0 -> 11.5 us, of 1083 x 1923 19.4 -> 11.6 us.  A sum
    of a constant over a cell's few points is counted in an integer."""
    from .hip_emit import KernelInfo, wrap_kernel
    from .expr_types import Float
    f = plan.func
    T = c_type(f.typ)
    nd = len(plan.fvars)
    od = sorted(plan.owned.values())
    z = plan.bin_dim
    others = [d for d in plan.free_dims if d != z]
    lo = dict((d, ceval_int(f.domain[d].lowerBound, {})) for d in plan.free_dims)
    ext = dict((d, ceval_int(f.domain[d].upperBound, {}) - lo[d] + 1) for d in plan.free_dims)
    G = (ext[z] + 1) // 2
    nthreads = 64
    ks = [plan.pre_size[rv] for rv in plan.rvars]
    w = lambda t, ind=1: L.append('  ' * ind + t)
    ncell = ' * '.join('(long long)%s' % exts[d] for d in od)
    w('const long long pmx_cell = (long long)pmx_tile * %d + (threadIdx.x >> 1);' % (nthreads // 2))
    w('const int pmx_h = (int)(threadIdx.x & 1) * %d;' % G)
    w('if (pmx_cell >= %s) return;' % ncell)
    w('long long cell = pmx_cell;')
    for d in reversed(od):
        w('const int c%d = (int)(cell %% %s) + (%s); cell /= %s;' % (d, exts[d], lbs[d], exts[d]))
    preimage()
    # one accumulator array per plane of the other free dims
    import itertools
    planes = list(itertools.product(*[range(lo[d], lo[d] + ext[d]) for d in others]))
    dflt = Value.numericToValue(f.default)
    known = dict((rc, _decided(plan, rc)) for rc in plan.cases)
    cases = [rc for rc in plan.cases if known[rc] is not False]

    def hits(pl):
        return [rc for rc in cases if tuple(
            ceval_int(rc.red.accumulate_ref.arguments[d], {}) for d in others) == pl]

    def counted(pl):
        """The constant a plane's only case sums, when counting gives the
        same bits."""
        h = hits(pl)
        if f.typ is not Float or len(h) != 1 or h[0].red.op_type != Op.Sum or \
                not (isinstance(dflt, Value) and isinstance(dflt.value, int)):
            return None
        v = Value.numericToValue(h[0].red.expression)
        if isinstance(v, Value) and isinstance(v.value, int) and \
                abs(v.value) * _prod_int(ks) + abs(dflt.value) <= 1 << 24:
            return v.value
        return None
    names = dict((d, 'c%d' % d) for d in od)
    for i, pl in enumerate(planes):
        if counted(pl) is not None:
            w('int a%d[%d];' % (i, G))
            w('for (int g = 0; g < %d; ++g) a%d[g] = 0;' % (G, i))
            continue
        nm = dict(names)
        nm.update(dict((d, str(v)) for d, v in zip(others, pl)))
        nm[z] = '(g + pmx_h + (%d))' % lo[z]
        dpr = Printer(dict((plan.fvars[d], nm[d]) for d in range(nd)), cb, mode, lazy=True)
        w('%s a%d[%d];' % (T, i, G))
        w('for (int g = 0; g < %d; ++g) a%d[g] = %s;' % (G, i, dpr.expr(f.default)))

    # f(r) = f0 + r / k along every variable: a cell that the domain's end
    # cuts has its points at fixed offsets too
    f0s = [plan.floor_start(rv, plan.cases[0].red.accumulate_ref.arguments[plan.owned[rv]],
                            f.reductionDomain[j].lowerBound) for j, rv in enumerate(plan.rvars)]

    # the reads of one point at affine indices that run at every point: what
    # a Case or a Select guards may lie outside its array elsewhere
    early = []
    for rc in cases:
        if known[rc] is None:
            continue
        for e in [rc.red.expression] + list(rc.red.accumulate_ref.arguments):
            for r in always_refs(e):
                if r.objectRef is not f and not any(a.has(Reference) for a in r.arguments if hasattr(a, 'has')):
                    text = cb(r, Printer(dict(zip(plan.rvars, rnames)), cb, mode, lazy=True), [])
                    if text not in [t for (t, _) in early]:
                        early.append((text, c_type(r.objectRef.typ)))
    at = ' + '.join('i%d * %d' % (j, _prod_int(ks[j + 1:])) for j in range(len(ks)))

    def cell(ind, point, inside=None):
        """All points of a cell, unrolled: their reads, then their updates.
        ``point(j)`` declares variable j's point from i<j>."""
        for n, (text, T_) in enumerate(early):
            w('%s pmx_x%d[%d];' % (T_, n, _prod_int(ks)), ind)
        for part in (0, 1):
            k = ind
            for j, kj in enumerate(ks):
                w('#pragma unroll', k)
                w('for (int i%d = 0; i%d < %d; ++i%d) { %s' % (j, j, kj, j, point(j)), k)
                k += 1
            if part == 0:
                for n, (text, _) in enumerate(early):
                    w('pmx_x%d[%s] = %s;' % (n, at, text), k)
            else:
                body(k, False, inside, dict((text, 'pmx_x%d[%s]' % (n, at)) for n, (text, _) in enumerate(early)))
            for j in ks:
                k -= 1
                w('}', k)
            if part == 0:
                # (otherwise the loads sink to their uses, to save registers,
                # and each row of the cell waits for memory)
                w('PMX_SCHED_BARRIER;', ind)

    def body(ind, owned, inside=None, regs=None):
        def rcb(ref, pr_, pro_):
            text = cb(ref, pr_, pro_)
            return (regs or {}).get(text, text)
        pr = Printer(dict(zip(plan.rvars, rnames)), rcb, mode, lazy=True)
        for rc in cases:
            tgt = rc.red.accumulate_ref.arguments
            pl = tuple(ceval_int(tgt[d], {}) for d in others)
            if pl not in planes:
                continue        # outside the grid
            i = planes.index(pl)
            w('{', ind)

            def target(d):
                pro = []
                q = pr.expr(tgt[d], pro)
                if classify_access(tgt[d], plan.rvars).kind == '*':
                    q = 'pmx_clampi(%s, %s, %s)' % (q, lbs[d], base.expr(f.domain[d].upperBound))
                for l in pro:
                    w(l, ind + 1)
                return q
            conds = []
            first = [] if known[rc] else _cond_dims(plan, rc)
            for d in first + ([d for d in od if d not in first] if owned else []):
                w('const int q%d = %s;' % (d, target(d)), ind + 1)
            if not known[rc]:
                vn = dict(zip(plan.rvars, rnames))
                for v, d in zip(plan.fvars, range(nd)):
                    if v not in plan.rvars:
                        vn[v] = 'q%d' % d
                cpro = []
                conds.append(Printer(vn, cb, mode, lazy=True).cond(rc.cond, cpro))
                for l in cpro:
                    w(l, ind + 1)
            if owned:
                conds += ['q%d == c%d' % (d, d) for d in od]
            if inside:
                conds.append(inside)
            if conds:
                w('const bool pmx_c = %s;' % ' && '.join(conds), ind + 1)
            # a condition guards the reads of the bin and of the value
            n = counted(pl)
            q = 'q%d' % z if z in first else target(z)
            w('const int pmx_z = %s - (%d) - pmx_h;' % (
                '(pmx_c ? %s : %d)' % (q, lo[z] - 2 * G) if conds else q, lo[z]), ind + 1)
            if n is None:
                pro = []
                val = pr.expr(rc.red.expression, pro)
                for l in pro:
                    w(l, ind + 1)
                w('const auto pmx_v = %s;' % (val if known[rc] else 'pmx_c ? (%s) : 0' % val), ind + 1)
            op = rc.red.op_type
            s = 'a%d[g]' % i
            upd = '%s += 1' % s if n is not None else \
                '%s = (%s + pmx_v)' % (s, s) if op == Op.Sum else \
                '%s = (%s * pmx_v)' % (s, s) if op == Op.Mul else \
                '%s = ((pmx_v %s %s)? (%s)(pmx_v): %s)' % (s, '<' if op == Op.Min else '>', s, T, s)
            w('#pragma unroll', ind + 1)
            w('for (int g = 0; g < %d; ++g) if (pmx_z == g) %s;' % (G, upd), ind + 1)
            w('}', ind)
    # whole pre-images: constant trip counts, all loads issued up front (the
    # order of the updates is the domain's)
    whole = ' && '.join('hi%d - lo%d + 1 == %d' % (j, j, k) for j, k in enumerate(ks))
    empty = ' || '.join('hi%d < lo%d' % (j, j) for j in range(len(ks)))
    if None not in f0s:
        # (a wavefront with a cut cell takes one path, not both in turn;
        # cells outside the domain take neither)
        w('if (PMX_ALL((%s) || %s)) {' % (whole, empty))
        w('if (%s) {' % whole, 2)
    else:
        w('if (%s) { {' % whole)
    cell(2, lambda j: 'const int r%d = lo%d + i%d;' % (j, j, j))
    if None not in f0s:
        # cut cells: the same points, those outside the domain read at its
        # nearest point and left out (a loop over the cell's own points
        # waits for every load in turn: 17 us of 1083 x 1923's grid)
        w('} } else if (!(%s)) {' % empty)
        cell(2, lambda j: 'const int p%d = (c%d - (%d)) * %d + i%d, r%d = pmx_clampi(p%d, %s, %s);'
             % (j, plan.owned[plan.rvars[j]], f0s[j], ks[j], j, j, j,
                base.expr(f.reductionDomain[j].lowerBound), base.expr(f.reductionDomain[j].upperBound)),
             ' && '.join('p%d == r%d' % (j, j) for j in range(len(ks))))
    else:
        w('} } else {')
        ind = 2
        for j in range(len(ks)):
            w('for (int r%d = lo%d; r%d <= hi%d; ++r%d) {' % (j, j, j, j, j), ind)
            ind += 1
        body(ind, True)
        for j in ks:
            ind -= 1
            w('}', ind)
    w('}')
    for i, pl in enumerate(planes):
        lin = None
        nm = dict(names)
        nm.update(dict((d, str(v)) for d, v in zip(others, pl)))
        nm[z] = '(g + pmx_h + (%d))' % lo[z]
        for d in range(nd):
            t = '(long long)(%s - (%s))' % (nm[d], lbs[d])
            lin = t if lin is None else '(%s * %s + %s)' % (lin, exts[d], t)
        n = counted(pl)
        val = 'a%d[g]' % i if n is None else '(%s)(%d + a%d[g] * %d)' % (T, dflt.value, i, n)
        w('#pragma unroll')
        w('for (int g = 0; g < %d; ++g) if (g + pmx_h < %d) G_%s[%s] = %s;' % (G, ext[z], f.name, lin, val))
    grid = '((%s + %d) / %d)' % (ncell, nthreads // 2 - 1, nthreads // 2)
    info = KernelInfo(kname, 'reduction', buffers, grid, nthreads, 0, plan, reads, [f])
    return [(wrap_kernel(kname, params, buffers, [f], nthreads, 0, L), info)]


_ATOMIC = {Op.Sum: 'atomicAdd', Op.Min: 'atomicMin', Op.Max: 'atomicMax'}


def _emit_atomic(pipe, plan, kname, mode, params, reads, buffers, exts, lbs, base, red_body, L):
    """Two kernels: ``<k>_init`` writes the default value at every target
    point, ``<k>`` runs one thread per reduction point (the domain
    flattened in its own order) and applies its value with a device
    atomic (a compare-and-swap loop for products)."""
    from .hip_emit import KernelInfo, wrap_kernel
    f = plan.func
    T = c_type(f.typ)
    nd = len(plan.fvars)
    nthreads = 256
    # init: one thread per target point
    I = []
    wi = lambda t, ind=1: I.append('  ' * ind + t)
    npts = ' * '.join('(long long)%s' % e for e in exts) or '1'
    wi('long long p = (long long)pmx_tile * %d + threadIdx.x;' % nthreads)
    wi('if (p >= %s) return;' % npts)
    wi('const long long lin = p;')
    for d in reversed(range(nd)):
        wi('const int f%d = (int)(p %% %s) + (%s); p /= %s;' % (d, exts[d], lbs[d], exts[d]))

    def cb(ref, pr, pro):
        g = ref.objectRef
        lin = None
        for d, arg in enumerate(ref.arguments):
            q = pr.expr(arg, pro)
            t = '(%s - (%s))' % (q, base.expr(g.domain[d].lowerBound))
            lin = t if lin is None else '(%s * %s + %s)' % (lin, _extent_c(g, d, base), t)
        return 'G_%s[%s]' % (g.name, lin or '0')
    dpr = Printer(dict((plan.fvars[d], 'f%d' % d) for d in range(nd)), cb, mode, lazy=True)
    pro = []
    dv = dpr.expr(f.default, pro)
    for l in pro:
        wi(l)
    wi('G_%s[lin] = (%s)(%s);' % (f.name, T, dv))
    init_name = kname + '_init'
    init_info = KernelInfo(init_name, 'reduction', [f], '((%s + %d) / %d)' % (npts, nthreads - 1, nthreads),
                           nthreads, 0, plan, [], [f])
    out = [(wrap_kernel(init_name, params, [f], [f], nthreads, 0, I), init_info)]
    # accumulation: one thread per reduction point
    del L[:]
    w = lambda t, ind=1: L.append('  ' * ind + t)
    rext = ['((%s) - (%s) + 1)' % (base.expr(iv.upperBound), base.expr(iv.lowerBound))
            for iv in f.reductionDomain]
    nred = ' * '.join('(long long)%s' % e for e in rext) or '1'
    w('long long p = (long long)pmx_tile * %d + threadIdx.x;' % nthreads)
    w('if (p >= %s) return;' % nred)
    for j in reversed(range(len(plan.rvars))):
        w('const int r%d = (int)(p %% %s) + (%s); p /= %s;' % (
            j, rext[j], base.expr(f.reductionDomain[j].lowerBound), rext[j]))
    tl = None
    for d in range(nd):
        t = '(long long)(q%d - (%s))' % (d, lbs[d])
        tl = t if tl is None else '(%s * %s + %s)' % (tl, exts[d], t)
    slot = 'G_%s[%s]' % (f.name, tl or '0')

    def update(op, val):
        v = '(%s)(%s)' % (T, val)
        if op in _ATOMIC:
            return '%s(&%s, %s);' % (_ATOMIC[op], slot, v)
        # product: compare-and-swap until no other thread intervened
        return ('{ %s* pa = &%s; const %s m = %s; %s old = *pa, seen; '
                'do { seen = old; old = atomicCAS(pa, seen, (%s)(seen * m)); } while (old != seen); }'
                % (T, slot, T, v, T, T))
    red_body(1, lambda: None, update)
    info = KernelInfo(kname, 'reduction', buffers, '((%s + %d) / %d)' % (nred, nthreads - 1, nthreads),
                      nthreads, 0, plan, reads, [f])
    out.append((wrap_kernel(kname, params, buffers, [f], nthreads, 0, L), info))
    return out
