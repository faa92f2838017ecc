"""Networks that one workgroup steps on its own: the resident step kernel.

A network without delays whose synapses all carry the same constant per pathway
(`on_pre: x += c`) and whose neurons fit a workgroup's registers needs no other
workgroup and no memory between its steps.  One workgroup per network runs any
number of steps in a launch:

* neuron q*T + x (thread x of T) keeps its state in thread x's registers, for
  q < R; the neurons beyond R*T (networks larger than the register file) keep
  theirs in memory;
* the spikes of a step go to a list in LDS (one LDS atomic per wave that has
  any);
* a spike's synapses are read from the CSR by source, 64 per wave, and counted
  per target and pathway in LDS (integer atomics, two 16-bit counts per word).
  Every event of a pathway applies the same operation with the same operand, so
  the count alone fixes the result: the owner applies the operation that many
  times at its next update, pathway by pathway in schedule order, which is the
  cython runtime's left fold over the queue
  (brian2/codegen/runtime/cython_rt/templates/synapses.pyx:42-50) bit for bit.

A step has one barrier (the spike list is complete) and, when there were spikes,
a second one (the counts are complete).
"""
import math
import re

from .chip import monitor_fields
from .codegen import ParamStruct, Renderer, source_header
from .kernels import _rename, group_block
from .kernels import heavy_operations as _heavy

LDS_BYTES = 163840       # LDS of one CU
STATE_REGISTERS = 80     # 32-bit registers of a thread that may hold neuron state
MAX_RESIDENT = 8         # neurons per thread in registers, at most
MAX_PATHWAYS = 4         # pathways of a network (two counts per LDS word)
UNITS_IN_FLIGHT = 4      # 64-synapse pieces a wave reads before it counts them
MAX_NEURONS = 65535      # spike lists hold 16-bit indices

_REFRACTORY = re.compile(r"not_refractory = \(bool\)\(\(hb_timestep\(\(double\)\(\(t - lastspike\)\), "
                         r"\(double\)\(dt\)\) >= ([\w.]+)\)\);")


def timestep_bound(k, dt):
    """The smallest y whose quotient int(y / dt) reaches k, for k >= 1 (hb_timestep's
    comparison with k).  y / dt rounds monotonically, so it is within a few units in the
    last place of k * dt."""
    y = k * dt
    while int(math.nextafter(y, 0.0) / dt) >= k:
        y = math.nextafter(y, 0.0)
    while int(y / dt) < k:
        y = math.nextafter(y, math.inf)
    return y


def releasable(k):
    """Whether the step at which a refractory period of k steps ends may be kept, in 32 bits and
    counted from a launch's first step (a longer period, of neurons that fire once say, is
    compared by its lastspike)."""
    return (k >= 1) & (k < 1 << 30)


def refractory_form(update, spike, var_types):
    """The name compared with in the refractoriness test `timestep(t - lastspike, dt) >= K`,
    when that test is the only use of lastspike and the only assignment of not_refractory
    in the lines of a neuron's update and spike; else None.

    The test is then true from one step on until the neuron's next spike: the kernel keeps
    that step instead of lastspike and not_refractory, compares integers, and forms the
    step anew only when the neuron spikes."""
    if var_types.get("lastspike") != "double" or var_types.get("not_refractory") != "bool":
        return None
    use = [ln for ln in list(update) + list(spike) if re.search(r"\blastspike\b|\bnot_refractory =[^=]", ln)]
    if len(use) != 1 or use[0] not in update or any("not_refractory" in ln for ln in spike):
        return None
    m = _REFRACTORY.fullmatch(use[0].strip())
    return None if m is None else m.group(1)


def neurons_in_registers(var_types):
    """Neurons per thread whose state the registers hold (1 to MAX_RESIDENT)."""
    words = sum(2 if ct in ("double", "long long") else 1 for ct in var_types.values())
    return max(1, min(MAX_RESIDENT, STATE_REGISTERS // max(1, words)))


class ResidentKernel:
    """Source of a resident step kernel.

    name        kernel name
    struct      its ParamStruct; fields used here: clock, step_off, dt, n_steps, status
    var_types   {state variable: C type}
    update      lines of one neuron's step: they read and write the variables by name and
                set hb_cond (the neuron spikes)
    spike       lines of a neuron that spikes (its reset), after the update
    refractory  whether a spike also sets not_refractory = false and lastspike = t
    pathways    [(variable, operator, C expression of the operand)] in schedule order
    prologue    lines that define, per workgroup: N, hb_off (the network's first neuron in
                the state arrays), hb_rp (row pointers by source), hb_step0
    event       lines that, for the synapse word hb_syn of source hb_src, define the target
                hb_tgt and the pathway's number hb_path
    events      further lines per event
    record      lines run for a step's spikes (s_spk[0 .. hb_nsp), any order) by every
                thread; may contain barriers
    begin/start lines that set hb_recq[hb_q] of neuron i, and lines run before its every step
                with hb_rec = hb_recq[hb_q] (state monitors; networks within the registers)
    finish      lines run once at the end by every thread
    resident    neurons per thread in registers
    bound       C expression of timestep_bound(K, dt) when K is the refractory period in
                steps and releasable, so that the release step may be kept (refractory_form)
    rows_in_lds, counts_in_lds   where row pointers and counts are kept

    What bounds it.  A step is a chain: the update of R neurons per thread, a barrier, the
    spikes' rows, their synapses (one memory round trip), LDS atomics, a barrier.  The update
    is straight-line code, so that a wave works on several neurons at a time: what few
    neurons need (a second event of a pathway, the spike itself) is tested once for all R
    and handled apart.  Measured on MI355X, cycles per step: a network of 7996 neurons
    (fp64, 16 waves, two spikes a step) 5070 for the update (2250 of them per wave alone;
    with branches per neuron 8000), 500 for the rows, 1150 for the synapses, 200 at the
    second barrier.  1024 networks of 500 to 8000 neurons: 42.9 -> 9.4 us per step against
    the state in memory and one spike's row at a time behind a barrier; 48 networks (fp32):
    9.5 -> 2.3.
    """

    def __init__(self, name, struct, var_types, update, pathways, prologue, event, spike=(), refractory=False,
                 record=(), start=(), begin=(), finish=(), events=(), max_threads=1024, resident=None,
                 rows_in_lds=True, counts_in_lds=True, shared=(), bound=None):
        if not 1 <= len(pathways) <= MAX_PATHWAYS:
            raise NotImplementedError(f"1 to {MAX_PATHWAYS} pathways")
        self.kernel_name, self.struct = name, struct
        self.words = W = (len(pathways) + 1) // 2
        self.resident = R = resident or neurons_in_registers(var_types)
        self.rows_in_lds, self.counts_in_lds = rows_in_lds, counts_in_lds
        period = refractory_form(update, spike, var_types) if refractory else None
        released = bound is not None and period is not None
        # what the registers hold: with the release step, neither lastspike nor not_refractory
        held = {v: ct for v, ct in var_types.items() if not (released and v in ("lastspike", "not_refractory"))}
        pt = {v: ("unsigned char" if ct == "bool" else ct) for v, ct in var_types.items()}
        load = {v: (f"p.a_{v}[hb_off + i] != 0" if ct == "bool" else f"p.a_{v}[hb_off + i]") for v, ct in var_types.items()}
        save = {v: (f"{v} ? 1 : 0" if ct == "bool" else v) for v, ct in var_types.items()}
        regs = ", ".join(f"r_{v}[hb_q]" for v in held)
        held_args, all_args = ", ".join(held), ", ".join(var_types)
        mem_load = " ".join(f"{ct} {v} = {load[v]};" for v, ct in var_types.items())
        mem_save = " ".join(f"p.a_{v}[hb_off + i] = ({pt[v]})({save[v]});" for v in var_types)
        # a neuron's events: counted by anybody, read and cleared by its owner (in memory: past
        # the caches, as the atomics go)
        pitch = "hb_np" if counts_in_lds else "N"
        at = f"s_cnt[(size_t){{w}} * {pitch} + i]"
        if counts_in_lds:
            read, clear = at, at + " = 0u;"
        else:
            read = f"(i < N ? __hip_atomic_load(&{at}, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0u)"
            clear = f"if (i < N) __hip_atomic_store(&{at}, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);"
        reads = [f"const unsigned int hb_c{w} = {read.format(w=w)};" for w in range(W)]
        clears = [clear.format(w=w) for w in range(W)]

        def decl(vs):
            return ", ".join(f"{ct}& {v}" for v, ct in vs.items())

        def field(r, c="hb_c{w}"):
            c = c.format(w=r // 2)
            return f"({c} & 0xffffu)" if r % 2 == 0 else f"({c} >> 16)"

        def each_event():  # every event of neuron i, pathway by pathway
            return [f"for (unsigned int n_ = {field(r)}; n_ > 0u; n_--) {var} {op} {val};"
                    for r, (var, op, val) in enumerate(pathways)]

        k = [source_header(max_threads), struct.c_decl()]
        k.append(f'extern "C" __global__ void __launch_bounds__({max_threads}) {name}(const {struct.name} p) {{')
        k += ["    " + x for x in prologue]
        k += [
            "    // the waves that the network's neurons fill: the others end here (barriers count the",
            "    // waves that run)",
            f"    const int NW = min((int)blockDim.x >> 6, max(1, (N + {64 * R - 1}) / {64 * R})), T = NW * 64;",
            "    if ((int)threadIdx.x >= T) return;",
            "    const int lane = threadIdx.x & 63;",
            "    const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));",
            "    const double dt = p.dt;",
            f"    const int hb_np = N > {R} * T ? N : {R} * T;  // counts of a pathway pair",
            "    extern __shared__ __align__(16) unsigned char hb_lds[];",
        ]
        lds = "hb_lds"
        if counts_in_lds:
            k.append(f"    unsigned int* const s_cnt = (unsigned int*)hb_lds;  // [{W}][hb_np], two counts a word")
            lds = f"(s_cnt + {W} * hb_np)"
        else:
            k.append(f"    unsigned int* const s_cnt = p.counts + (size_t)hb_off * {W};")
        if rows_in_lds:
            k.append(f"    unsigned int* const s_rp = (unsigned int*){lds};")
            lds = "(s_rp + N + 1)"
        row = "s_rp[{}]" if rows_in_lds else "hb_rp[{}]"
        k += [
            f"    unsigned short* const s_spk = (unsigned short*){lds};",
            "    __shared__ int s_n[3];  // spikes of steps hb_s % 3: added to, read, cleared in turn",
        ]
        k += ["    " + x for x in shared]
        if released:
            k += [
                f"    const double hb_tb = {bound};",
                "    // a neuron that last spiked at time x is not refractory from the step k on (a double:",
                "    // exact) at which (k * dt - x) + 1e-3 * dt >= hb_tb, which grows with k",
                "    auto hb_free = [&](const double x, const double k) { return (k * dt - x) + 1e-3 * dt >= hb_tb; };",
                "    auto hb_release = [&](const double x) {  // that step, counted from hb_step0 and 0 at least",
                "        const double k0 = (double)hb_step0;",
                "        if (hb_free(x, k0)) return 0;",
                "        double k = floor((hb_tb + x) / dt);",
                "        for (int j = 0; j < 8 && hb_free(x, k - 1.0); j++) k -= 1.0;",
                "        for (int j = 0; j < 8 && !hb_free(x, k); j++) k += 1.0;",
                "        k -= k0;",
                "        return k < 2147483647.0 ? (int)k : 0x7fffffff;",
                "    };",
            ]
        # the update of a neuron in registers, and of one in memory where they differ
        for fn, vs in (("hb_update", held), ("hb_update_mem", var_types)):
            reg = released and fn == "hb_update"
            lines = ["not_refractory = hb_s >= hb_rel;" if reg and _REFRACTORY.fullmatch(x.strip()) else x for x in update]
            k += [
                "    // one step of neuron i after the events of the step before: whether it spikes",
                f"    auto {fn} = [&](const int i, const int hb_s, const double t, {decl(vs)}"
                f"{', const int hb_rel' if reg else ''}) __attribute__((always_inline)) {{",
                "        const int _idx = i;",
                "        (void)_idx; (void)hb_s; (void)t;",
                "        bool hb_cond = false;",
            ]
            k += ["        bool not_refractory;"] if reg else []
            k += ["        " + x for x in lines]
            k += ["        return hb_cond;", "    };"]
            if not released:
                break
        k += [f"    auto hb_spike = [&](const int i, const double t, {decl(held)}) __attribute__((always_inline)) {{",
              "        const int _idx = i;", "        (void)_idx; (void)t;"]
        if refractory and not released:
            k.append("        not_refractory = false; lastspike = t;")
        k += ["        " + x for x in spike]
        k.append("    };")
        if rows_in_lds:
            k.append("    for (int i = threadIdx.x; i <= N; i += T) s_rp[i] = hb_rp[i];")
        k.append("    if (threadIdx.x < 3) s_n[threadIdx.x] = 0;")
        first = "hb_release(p.a_lastspike[hb_off + i])"
        if released and counts_in_lds:  # formed one by one (the code is long), passed through the counts
            k += [
                "    #pragma unroll 1",
                f"    for (int i = threadIdx.x; i < {R} * T; i += T)",
                f"        s_cnt[i] = i < N ? (unsigned int){first} : 0x7fffffffu;",
            ]
            first = "(int)s_cnt[i]"
        for v, ct in held.items():
            k.append(f"    {ct} r_{v}[{R}];")
        if released:
            k.append(f"    int hb_rels[{R}];")
        if start:
            k.append(f"    int hb_recq[{R}];")
        k += [
            f"    unsigned long long hb_act[{R}];  // lanes with a neuron (scalars)",
            "    #pragma unroll",
            f"    for (int hb_q = 0; hb_q < {R}; hb_q++) {{",
            "        const int i = hb_q * T + (int)threadIdx.x;",
            "        const bool act = i < N;",
            "        hb_act[hb_q] = __builtin_amdgcn_ballot_w64(act);",
        ]
        for v, ct in held.items():
            k.append(f"        r_{v}[hb_q] = act ? {load[v]} : ({ct})0;")
        if released:
            k.append(f"        hb_rels[hb_q] = act ? {first} : 0x7fffffff;")
        k += ["        " + x for x in begin]
        k.append("        // waited for here: a wait inside the loop would be for the step's stores as well")
        k += [f'        asm volatile("" : "+v"(r_{v}[hb_q]));' for v, ct in held.items() if ct != "bool"]
        k.append("    }")
        if counts_in_lds:
            k.append(f"    for (int i = threadIdx.x; i < {W} * hb_np; i += T) s_cnt[i] = 0u;")
        k.append("    __syncthreads();")
        fence = [] if counts_in_lds else ["__threadfence();  // the counts are in memory"]
        put = [
            "if (b_ != 0ull) {  // the wave's spikes to the list",
            "    int o_ = 0;",
            "    if (lane == 0) o_ = atomicAdd(&s_n[hb_cur], __popcll(b_));",
            "    o_ = __builtin_amdgcn_readfirstlane(o_);",
            "    if ((b_ >> lane) & 1ull) {",
            "        s_spk[o_ + __popcll(b_ & ((1ull << lane) - 1ull))] = (unsigned short)i;",
        ]
        k += [
            "    int hb_cur = 0, hb_old = 2;",
            "    double hb_k = (double)hb_step0;  // the step (exact)",
            "    for (int hb_s = 0; hb_s < p.n_steps; hb_s++, hb_k += 1.0) {",
            "        const long long hb_step = hb_step0 + hb_s;",
            "        const double t = hb_k * dt;  // (double)hb_step * dt",
            "        (void)hb_step;",
        ]
        k += [f"        unsigned int hb_c{w}[{R}], hb_o{w} = 0u;" for w in range(W)]
        k += ["        #pragma unroll", f"        for (int hb_q = 0; hb_q < {R}; hb_q++) {{  // all reads in flight together",
              "            const int i = hb_q * T + (int)threadIdx.x;"]
        k += [f"            hb_c{w}[hb_q] = {read.format(w=w)};" for w in range(W)]
        k += [f"            hb_o{w} |= hb_c{w}[hb_q];" for w in range(W)]
        k.append("        }")
        more = " | ".join(f"(hb_o{w} & 0xfffefffeu)" for w in range(W))
        same = len({v for v, _, _ in pathways}) < len(pathways)
        # pathways into one variable follow each other, so only the last of them may leave its
        # last event to the selection below
        last = {v: r for r, (v, _, _) in enumerate(pathways)}
        rest = " | ".join(f"hb_o{w}" for w in range(W)) if same else more
        k += [f"        if (__builtin_amdgcn_ballot_w64(({rest}) != 0u) != 0ull) {{  // more events than one of a pathway",
              "            #pragma unroll", f"            for (int hb_q = 0; hb_q < {R}; hb_q++) {{"]
        k += [f"                {held[v]}& {v} = r_{v}[hb_q];" for v in dict.fromkeys(v for v, _, _ in pathways)]
        for r_, (var, op, val) in enumerate(pathways):
            k.append(f"                for (unsigned int n_ = {field(r_, 'hb_c{w}[hb_q]')}; n_ > "
                     f"{1 if last[var] == r_ else 0}u; n_--) {var} {op} {val};")
        k += ["            }", "        }",
              f"        unsigned long long hb_b[{R}], hb_any = 0ull;  // the wave's spikes (scalars)",
              "        #pragma unroll",
              f"        for (int hb_q = 0; hb_q < {R}; hb_q++) {{  // lanes without a neuron compute on zeros",
              "            const int i = hb_q * T + (int)threadIdx.x;"]
        for r_, (var, op, val) in enumerate(pathways):
            if last[var] == r_:
                k += [f"            {{ {held[var]} x_ = r_{var}[hb_q]; x_ {op} {val}; "
                      f"r_{var}[hb_q] = {field(r_, 'hb_c{w}[hb_q]')} != 0u ? x_ : r_{var}[hb_q]; }}"]
        k += ["            " + x for x in clears]
        if start:
            k += ["            if (i < N) {"] + [f"                const {ct}& {v} = r_{v}[hb_q];" for v, ct in held.items()]
            k += ["                const int hb_rec = hb_recq[hb_q];"]
            k += ["                " + x for x in start] + ["            }"]
        k += [
            f"            hb_b[hb_q] = __builtin_amdgcn_ballot_w64(hb_update(i, hb_s, t, {regs}"
            f"{', hb_rels[hb_q]' if released else ''})) & hb_act[hb_q];",
            "            hb_any |= hb_b[hb_q];",
            "        }",
            "        if (hb_any != 0ull) {",
            "            int hb_x = (int)threadIdx.x;  // hidden: see the end",
            '            asm volatile("" : "+v"(hb_x));',
        ]
        if released:
            k += [
                "            // the release step of a neuron that spikes now: K steps on, or one beside it by rounding",
                f"            const double k_ = hb_k + (double)({period});",
                f"            const int rel_ = hb_s + (int)({period}) + (hb_free(t, k_ - 1.0) ? -1 : hb_free(t, k_) ? 0 : 1);",
            ]
        k += ["            #pragma unroll", f"            for (int hb_q = 0; hb_q < {R}; hb_q++) {{",
              "                const int i = hb_q * T + hb_x;", "                const unsigned long long b_ = hb_b[hb_q];"]
        k += ["                " + x for x in put]
        if released:
            k.append("                        hb_rels[hb_q] = rel_; p.a_lastspike[hb_off + i] = t;")
        k += [f"                        hb_spike(i, t, {regs});", "                    }", "                }",
              "            }", "        }",
              f"        for (int j0 = {R} * T; j0 < N; j0 += T) {{  // neurons beyond the registers",
              "            const int i = j0 + (int)threadIdx.x;",
              "            bool hb_sp = false;",
              "            if (i < N) {",
              f"                {mem_load}"]
        k += ["                " + x for x in reads + each_event() + clears]
        k += [f"                hb_sp = {'hb_update_mem' if released else 'hb_update'}(i, hb_s, t, {all_args});",
              "                if (hb_sp) {"]
        if released:
            k.append("                    not_refractory = false; lastspike = t;")
        k += [f"                    hb_spike(i, t, {held_args});", "                }",
              f"                {mem_save}", "            }",
              "            const unsigned long long b_ = __builtin_amdgcn_ballot_w64(hb_sp);"]
        k += ["            " + x for x in put] + ["                }", "            }"]
        k += ["        }"] + ["        " + x for x in fence] + [
            "        __syncthreads();",
            "        const int hb_nsp = s_n[hb_cur];",
            "        // the last step's counter: every wave has read it, and it is added to again only",
            "        // behind the next step's barrier",
            "        if (threadIdx.x == 0) s_n[hb_old] = 0;",
            "        hb_old = hb_cur;",
            "        hb_cur = hb_cur == 2 ? 0 : hb_cur + 1;",
            "        if (hb_nsp > 0) {",
        ]
        k += ["            " + x for x in record]

        def unit(u, ok, x, src, ind):
            return [ind + ln for ln in (
                f"const int l_ = __builtin_ctzll(__builtin_amdgcn_ballot_w64(in_ > {u}));",
                "const int first_ = __builtin_amdgcn_readlane(in_ - nu_, l_);",
                "const unsigned int a_ = (unsigned int)__builtin_amdgcn_readlane((int)ra_, l_);",
                "const unsigned int z_ = (unsigned int)__builtin_amdgcn_readlane((int)rb_, l_);",
                f"{src} = __builtin_amdgcn_readlane(sp_, l_);",
                f"const unsigned int e_ = a_ + (unsigned int)({u} - first_) * 64u + (unsigned int)lane;",
                f"{ok} = e_ < z_;",
                f"{x} = p.post[e_ < z_ ? e_ : z_ - 1u];",
            )]

        def count(x, src, ind):
            return [ind + ln for ln in (
                f"const unsigned int hb_syn = {x};", f"const int hb_src = {src};", "(void)hb_src;", *event,
                f"atomicAdd(&s_cnt[(hb_path >> 1) * {pitch} + hb_tgt], hb_path & 1 ? 0x10000u : 1u);", *events)]

        F = UNITS_IN_FLIGHT
        k += [
            "            // 64 spikes at a time: lane l holds spike l's row; the rows' pieces of 64 synapses",
            "            // are dealt to the waves",
            "            for (int c0 = 0; c0 < hb_nsp; c0 += 64) {",
            "                const int sp_ = c0 + lane < hb_nsp ? (int)s_spk[c0 + lane] : -1;",
            f"                const unsigned int ra_ = sp_ >= 0 ? {row.format('sp_')} : 0u, "
            f"rb_ = sp_ >= 0 ? {row.format('sp_ + 1')} : 0u;",
            "                const int nu_ = (int)((rb_ - ra_ + 63u) >> 6);",
            "                const int in_ = hb_wave_incl_scan(nu_);",
            "                const int U = __builtin_amdgcn_readlane(in_, 63);",
            "                if (U <= NW) {  // at most one piece per wave",
            "                    if (wid < U) {",
            "                        int g_; bool ok_; unsigned int x_;",
        ]
        k += unit("wid", "ok_", "x_", "g_", " " * 24)
        k += ["                        if (ok_) {"] + count("x_", "g_", " " * 28) + ["                        }"]
        k += [
            "                    }",
            "                } else {",
            f"                    for (int u0 = wid; u0 < U; u0 += {F} * NW) {{",
            f"                        unsigned int x_[{F}];",
            f"                        int g_[{F}];",
            f"                        bool ok_[{F}];",
            "                        #pragma unroll",
            f"                        for (int j = 0; j < {F}; j++) {{",
            "                            const int u = u0 + j * NW;",
            "                            ok_[j] = false; x_[j] = 0u; g_[j] = 0;",
            "                            if (u < U) {  // the same for the wave",
        ]
        k += unit("u", "ok_[j]", "x_[j]", "g_[j]", " " * 32)
        k += [
            "                            }",
            "                        }",
            "                        #pragma unroll",
            f"                        for (int j = 0; j < {F}; j++)",
            "                            if (ok_[j]) {",
        ]
        k += count("x_[j]", "g_[j]", " " * 32)
        k += [
            "                            }",
            "                    }",
            "                }",
            "            }",
        ] + ["            " + x for x in fence] + [
            "            __syncthreads();",
            "        }",
            "    }",
            "    // the last step's events, and the state back to memory (the index is hidden from the",
            "    // compiler, which would keep the addresses of the first loads in registers for it)",
            "    int hb_x = (int)threadIdx.x;",
            '    asm volatile("" : "+v"(hb_x));',
            "    #pragma unroll",
            f"    for (int hb_q = 0; hb_q < {R}; hb_q++) {{",
            "        const int i = hb_q * T + hb_x;",
            "        if (i < N) {",
        ]
        k += ["            " + x for x in reads]
        k += [f"            {held[v]}& {v} = r_{v}[hb_q];" for v in dict.fromkeys(v for v, _, _ in pathways)]
        k += ["            " + x for x in each_event() + clears]
        for v, ct in held.items():
            val = f"r_{v}[hb_q] ? 1 : 0" if ct == "bool" else f"r_{v}[hb_q]"
            k.append(f"            p.a_{v}[hb_off + i] = ({pt[v]})({val});")
        if released:
            k.append("            p.a_not_refractory[hb_off + i] = p.n_steps - 1 >= hb_rels[hb_q] ? 1 : 0;")
        k += [
            "        }",
            "    }",
            f"    for (int i = {R} * T + hb_x; i < N; i += T) {{",
            f"        {mem_load}",
        ]
        k += ["        " + x for x in reads + each_event() + clears]
        k += [f"        {mem_save}", "    }"]
        k += ["    " + x for x in finish]
        k.append("}")
        self.source = "\n".join(k) + "\n"

    def lds_bytes(self, N, threads, extra=0):
        """Dynamic LDS of a workgroup of that many threads for a network of N neurons."""
        b = 2 * N + extra
        if self.counts_in_lds:
            b += 4 * self.words * max(N, self.resident * threads)
        if self.rows_in_lds:
            b += 4 * (N + 1)
        return (b + 15) // 16 * 16


def lds_plan(N, words, extra=0):
    """(rows_in_lds, counts_in_lds) for networks of up to N neurons: the counts first (they
    are written), then the row pointers (read, once per spike)."""
    room = LDS_BYTES - 2048 - 2 * N - extra
    c = 4 * words * max(N, 1024 * MAX_RESIDENT)
    counts = c <= room
    rows = counts and c + 4 * (N + 1) <= room
    return rows, counts


def heavy_operations(specs):
    """Exponentials, powers and the like in the vector code of code objects."""
    return sum(max(_heavy(e) for e in [e for _, e in st.get("bool_exprs") or []] or [st["expr"]])
               for spec in specs for st in (spec.vector if spec is not None else ()))


def plain_network(net, groups, paths, summed):
    """Whether Network net is one group with synapses onto itself whose events are no more than
    their number: no delays, no variables of the synapses; default launch shapes."""
    if len(groups) != 1 or summed or not 1 <= len(paths) <= MAX_PATHWAYS:
        return False
    if any(x is not None for x in (net.tile, net.npt, net.gather_pairs, net.bucket_cap)):
        return False
    g = groups[0]
    if getattr(g, "su", None) is None or g.N < 1:
        return False
    for s in paths:
        if s.source is not g or s.target is not g or s.syn_vars or s.plastic or s.post_spec is not None:
            return False
        if s.count_events or s.carry is not None or s.csr["dmin"] != 0 or s.csr["n_seg"] != 1:
            return False
        if len(s.spec.vector) != 1 or g.vars[s.target_var] not in ("double", "float"):
            return False
    return True


class GroupStep:
    """The resident step of a neuron group with synapses onto itself (Network's small
    networks): the ResidentKernel with the group's monitors.

    group      its NeuronGroup; scalars {(tag, name): (value, ctype)} of its code objects
    pathways   [(Synapses, {name: (value, ctype)})] in schedule order
    val_t      type in which the pathways' values are held before they are applied"""

    MAX_SYNAPSES = 1 << 25
    # heavy operations of an update, and neurons x these, from which steps over the whole chip
    # are faster; neurons x these from which staged launches are
    CHIP_HEAVY = 8
    CHIP_WORK = {"double": 1024, "float": 2560}
    MAX_HEAVY = {"double": 16384, "float": 36864}

    def __init__(self, group, scalars, pathways, val_t, n_syn, dt):
        g = group
        # as few neurons per thread as 1024 threads allow: 500 neurons one / two / eight per
        # thread 0.81 / 1.07 / 1.62 us per step, 4000 four / eight 2.03 / 2.39
        self.rows = -(-g.N // 1024)
        waves = -(-g.N // 64)
        self.threads = 64 * -(-waves // self.rows)
        ps = ParamStruct(f"hbr_{g.name}")
        ps.ptr("clock", "long long")
        ps.val("step_off", "long long")
        ps.val("dt", "double")
        ps.val("n_steps", "int")
        ps.val("N", "int")
        for v, ct in g.vars.items():
            ps.ptr(f"a_{v}", "unsigned char" if ct == "bool" else ct)
        for (tg, n), (_, ct) in sorted(scalars.items()):
            ps.val(f"{tg}_{n}", ct)
        for r, (_, sc) in enumerate(pathways):
            for n, (_, ct) in sorted(sc.items()):
                ps.val(f"c{r}_{n}", ct)
        ps.val("bound", "double")
        ps.ptr("row_ptr", "unsigned int", const=True)
        ps.ptr("post", "unsigned int", const=True)
        ps.ptr("events", "unsigned long long")
        ps.ptr("counts", "unsigned int")
        ps.ptr("status", "int")
        monitor_fields(ps, g)
        self.struct = ps

        def block(tag, spec, extra=()):
            return group_block(tag, spec, g.vars, scalars, g.float_t, extra, select=True)

        update, spike = [], []
        if g.su is not None:
            update += ["{"] + block("su", g.su) + ["}"]
        if g.th is not None:
            update += ["{"] + block("th", g.th, {"_cond": "bool"}) + ["hb_cond = _cond;", "}"]
        if g.rs is not None:
            spike = block("rs", g.rs)
        # the refractory period in steps, compared through its bound
        recorded = set(g.stmon.variables) if g.stmon else set()
        self.bound = None
        name = refractory_form(update, spike, g.vars)
        if name is not None and not recorded & {"lastspike", "not_refractory"}:
            value, ct = scalars.get(("su", name[len("p.su_"):]), (0, None))
            if ct == "long long" and releasable(value):
                self.bound = timestep_bound(value, dt)
        ops, events = [], []
        for r, (s, sc) in enumerate(pathways):
            c, _ = Renderer({n: ct for n, (_, ct) in sc.items()}).render(s.spec.vector[0]["expr"])
            c, = _rename([c], {n: f"p.c{r}_{n}" for n in sc})
            ops.append((s.target_var, s.op, f"(({val_t})({c}))"))
            events.append(f"hb_ev{r} += hb_path == {r} ? 1u : 0u;")
        prologue = [
            "const int N = p.N, hb_off = 0;",
            "const unsigned int* hb_rp = p.row_ptr;",
            "const long long hb_step0 = p.clock[0] + p.step_off;",
        ] + [f"unsigned long long hb_ev{r} = 0ull;" for r in range(len(ops))]
        record, finish, shared, begin, start = [], [], [], [], []
        # the record is the last waves' work: the first ones have the spikes' synapses
        each = "for (int j = T - 1 - (int)threadIdx.x; j < {n}; j += T) {{"
        if g.smon:
            add = ["if (o_ < (unsigned long long)p.mon_cap) { p.mon_i[o_] = id_; p.mon_step[o_] = (int)hb_step; }",
                   "atomicAdd(&p.mon_count[id_ - p.mon_start], 1);"]
            if g.smon.range == (0, g.N):
                prologue.append("unsigned long long hb_mn = p.mon_n[0];")
                record += [each.format(n="hb_nsp"), "    const int id_ = (int)s_spk[j];",
                           "    const unsigned long long o_ = hb_mn + (unsigned long long)j;"]
                record += ["    " + x for x in add] + ["}", "hb_mn += (unsigned long long)hb_nsp;"]
            else:
                prologue.append("const unsigned long long hb_m0 = p.mon_n[0];")
                shared += ["__shared__ unsigned int s_mon;  // records of the launch", "if (threadIdx.x == 0) s_mon = 0u;"]
                record += [each.format(n="hb_nsp"), "    const int id_ = (int)s_spk[j];",
                           "    if (id_ >= p.mon_start && id_ < p.mon_stop) {",
                           "        const unsigned long long o_ = hb_m0 + (unsigned long long)atomicAdd(&s_mon, 1u);"]
                record += ["        " + x for x in add] + ["    }", "}"]
                finish += ["const unsigned long long hb_mn = hb_m0 + (unsigned long long)s_mon;"]
            finish += ["if (threadIdx.x == 0) {", "    p.mon_n[0] = hb_mn;",
                       "    if (hb_mn > (unsigned long long)p.mon_cap) atomicOr(p.status, 2);", "}"]
        if g.rmon:
            record += [
                "if (p.rate_cnt && hb_step - p.rate_row0 >= 0 && hb_step - p.rate_row0 < p.rate_rows) {",
                "    " + each.format(n="hb_nsp"),
                "        const int id_ = (int)s_spk[j];",
                "        if (id_ >= p.rate_start && id_ < p.rate_stop) atomicAdd(&p.rate_cnt[hb_step - p.rate_row0], 1);",
                "    }",
                "}",
            ]
        if g.stmon:  # recorded neurons: their place in rec_idx, or -1
            begin += [
                "hb_recq[hb_q] = -1;",
                "if (act) {",
                "    int lo = 0, hi = p.n_rec;",
                "    while (lo < hi) { const int m = (lo + hi) >> 1; if (p.rec_idx[m] < i) lo = m + 1; else hi = m; }",
                "    if (lo < p.n_rec && p.rec_idx[lo] == i) hb_recq[hb_q] = lo;",
                "}",
            ]
            nv = len(g.stmon.variables)
            start += ["if (hb_rec >= 0 && hb_step - p.rec_row0 >= 0 && hb_step - p.rec_row0 < p.rec_rows) {",
                      f"    double* const o_ = p.rec_buf + (size_t)(hb_step - p.rec_row0) * {nv} * p.n_rec + hb_rec;"]
            start += [f"    o_[(size_t){a} * p.n_rec] = (double){v};" for a, v in enumerate(g.stmon.variables)] + ["}"]
        finish += [f"if (hb_ev{r}) atomicAdd(&p.events[{r}], hb_ev{r});" for r in range(len(ops))]
        finish.append("if (threadIdx.x == 0) p.clock[0] = hb_step0 + p.n_steps;")
        self.ops, self.n_syn = ops, n_syn
        self.kernel = ResidentKernel(
            f"resident_{g.name}", ps, g.vars, update, ops, prologue,
            ["const int hb_tgt = (int)(hb_syn & 0xffffu);", "const int hb_path = (int)(hb_syn >> 16);"], spike=spike,
            refractory=g.uses_refractory and g.th is not None, record=record, start=start, begin=begin, finish=finish,
            events=events, max_threads=self.threads, resident=self.rows, shared=shared,
            bound="p.bound" if self.bound is not None else None)
        self.lds_bytes = self.kernel.lds_bytes(g.N, self.threads)

    @classmethod
    def too_heavy(cls, groups):
        """Whether the only group's update is rather for the whole chip (see takes)."""
        g = groups[0] if len(groups) == 1 else None
        if getattr(g, "su", None) is None:
            return False
        heavy = heavy_operations((g.su, g.th, g.rs))
        return heavy >= cls.CHIP_HEAVY or g.N * heavy > cls.CHIP_WORK[g.float_t]

    @classmethod
    def takes(cls, net, groups, paths, summed):
        """Whether Network net is stepped this way: one group whose neurons fit a workgroup's
        registers, synapses from it onto itself without delays or variables of their own,
        default launch shapes, an update that one compute unit can carry.

        Measured on MI355X, us per step, against a launch for the group and one per pathway: CUBA
        with 500 / 4000 / 8192 neurons 0.84 / 2.2 / 3.9 against 12.3 / 15.7 / 18.0; 8000 neurons
        with 19 million synapses 3.9 (in a volley one compute unit has all the events, hence the
        bound on them); over the whole chip (chip.ChipSteps) 1.7 / 3.1 / 3.8.  An update with
        exponentials is throughput, and latency where the waves are few: COBAHH (29 of them)
        with 20 / 100 / 400 / 1000 neurons 7.7 / 8.1 / 15.6 / 49.8 against 4.0 / 4.0 / 4.9 / 5.1
        over the whole chip in fp64, 3.9 / 4.5 / 6.3 / 15.6 against 2.8 / 2.8 / 3.6 / 3.9 in
        fp32: 0.2 us per heavy operation of a wave, 1.7 (fp64) and 0.5 per 1000 neurons
        (too_heavy).  Networks that cannot count their events that way (a pair with two
        synapses) are staged otherwise: 400 / 600 neurons 15.8 / 31.8 against 22.7 / 24.2 in
        fp64, 1000 neurons 15.7 against 22.4 in fp32."""
        if not plain_network(net, groups, paths, summed):
            return False
        g = groups[0]
        if g.N > 1024 * neurons_in_registers(g.vars):
            return False
        if g.N * heavy_operations((g.su, g.th, g.rs)) > cls.MAX_HEAVY[g.float_t]:
            return False
        return sum(int(s.csr["n_syn"]) for s in paths) <= cls.MAX_SYNAPSES

    @staticmethod
    def merged_rows(group, paths):
        """The pathways' synapses as one CSR by source: row pointers and, per synapse, the
        target and the pathway's number (bits 16 and up).  None when a target has more than
        65535 synapses of a pathway (its count would not fit)."""
        import torch

        N, words, src = group.N, [], []
        for r, s in enumerate(paths):
            ptr = s.csr["seg_ptr"].long()
            a = s.src_range[0]
            n = int(s.csr["n_syn"])
            post = s.csr["post"][:n]
            if n > 65535 and int(torch.bincount(post, minlength=N).max()) > 65535:
                return None
            words.append(post | (r << 16))
            src.append(torch.repeat_interleave(torch.arange(a, a + len(ptr) - 1, device=post.device), ptr[1:] - ptr[:-1],
                                               output_size=n))
        src, words = torch.cat(src), torch.cat(words)
        order = torch.argsort(src, stable=True)
        rows = torch.zeros(N + 1, dtype=torch.int64, device=src.device)
        rows[1:] = torch.bincount(src, minlength=N).cumsum(0)
        post = words[order] if len(words) else torch.zeros(1, dtype=torch.int32, device=src.device)
        return rows.int(), post.int().contiguous()
