// Line solvers that generate the stencils of the primary operator from the
// slab material while they walk their lines (march grids periodic along both
// axes).
//
// The mu*R stencils of a point are 40 real and 12 walk-off values, all of them
// products of nine fields of the slab average (1/eps_zz, K, sqrt(K)^-1, v) at
// the point and its neighbours.  Stored, they are 640 bytes a point in FP64
// (written once and read 15-21 complex planes at a time by each of the six
// solver launches of a slab); the nine fields are 72.  A solver thread walks
// the consecutive points of its chunk along the line, with the fields of the
// last two rows in registers, so that the right-hand side, the tridiagonal row
// and the elimination of a point follow each other.
//
// The block walks in step: at step j every chunk is at its row j, and the rows
// of all chunks (W + 2 columns of material and fields) come through LDS,
// loaded straight into it two steps ahead.  Loaded row by row by the threads
// themselves, each row cost a round trip to the Infinity Cache (512^2, one
// propagation pair: 37-49 us a launch).
//
// What bounds it: at one propagation pair on 512^2 two waves per SIMD, one of
// each component, FP64 arithmetic about half of the time (200 instructions a
// row of the two) and 81 MB of traffic a launch; at 64^2 the chain of steps
// and cyclic reductions.  Device time per launch, MI355X, against the solvers
// on stored stencils (x / y lines): 512^2 x 1 pair 22-23 us (29-36 / 35),
// 1024^2 120-125 us (130-156 / 225-238).  Per slab, whole march: 64^2 54 us
// (68), 161^2 74 us (96), 128^2 x 7 pairs 109 us (120), x 147 pairs 1.27 ms
// (1.46), 256^2 x 147 pairs 5.5 ms (6.2).  A whole 512^2 x 100 propagation
// 25.1 -> 17.3 ms, 1024^2 x 200 267.5 -> 172.7 ms.
//
// Lanes of a wave lie across the lines (consecutive in memory) and chunks of
// them: the state is kept with the line axis slow, [l][t] for lines along l.
// The lines of the two half-steps run along different axes, so the last
// launch of a half-step writes its result through LDS in the other order.
//
// Everything is written once in (l, t) terms, l along the line and t across
// it: exchanging x and y exchanges the two field components and the xx / yy
// members of the material, and the operators
//   A_t = [T_ll T_lt; T_tl+C_tl T_tt+C_tt]      (explicit half, along t)
//   O_l = [C_ll L_lt+C_lt; L_tl 0]              (Neumann coupling)
// of lines along l (L, T: stencils along l and t, C: corners) are the x and
// the y half-step's for l = x and l = y
// (ParaxialPrimaryEvolutionOperator.cpp:102-210, 212-490).
#include <stdexcept>
#include <string>
#include <type_traits>

#include "kernels.h"
#include "walk.h"

namespace nmk {

#define NMK_WALK_CHECK()                                                                         \
    do {                                                                                         \
        hipError_t e_ = hipGetLastError();                                                       \
        if (e_ != hipSuccess) throw std::runtime_error(std::string("HIP launch failed: ") +     \
                                                       hipGetErrorString(e_));                   \
    } while (0)

namespace {

// 1/v: the hardware estimate and two Newton steps (an IEEE division is twice
// as long a chain, and the eliminations are chains of them: 64^2 x 20 1.106 ms
// against 1.125, 1024^2 x 200 172.7 against 173.9); the fix-up gives the special
// values of the division.  Errors of nine marches (64^2 to 300 x 210, droplets,
// beams, oblique) against long double arithmetic: equal to four digits.
__device__ __forceinline__ double rcp_newton(double v) {
    double r = __builtin_amdgcn_rcp(v);
    r = fma(r, fma(-v, r, 1.0), r);
    r = fma(r, fma(-v, r, 1.0), r);
    return __builtin_amdgcn_div_fixup(r, v, 1.0);
}
__device__ __forceinline__ c64 wrcp(c64 a) {
    const double r = rcp_newton(a.x * a.x + a.y * a.y);
    return {a.x * r, -a.y * r};
}

// material of one point in (l, t) terms
struct Mat {
    double kll, klt, ktt, ill, ilt, itt, e, vt, vl;
};

// the parts of the material a right-hand side reads at the side columns t -+ 1
// and whether it reads the fields there
//   first launch (NEU 0): both components, the transverse one with its walk-off
//   Neumann launches: the line component only
template <int NEU, int COMP>
struct Uses {
    static constexpr bool side = NEU == 0 || COMP == 0;
    static constexpr bool side_v = NEU == 0 && COMP == 1;
    static constexpr bool corner = NEU == 0 ? COMP == 1 : COMP == 0;
    // fields of the line's own column
    static constexpr bool own_l = !(NEU == 1 && COMP == 0), own_t = !(NEU == 1 && COMP == 1);
};

// one point of the block's rows in LDS
__device__ __forceinline__ Mat mat_of(const c64 *v) {
    const c64 a = v[0], b = v[1], c = v[2], d = v[3], e = v[4];
    return Mat{a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y, e.x};
}

// LDS rows of a step, 16-byte units: W + 2 points of material (5 units each) of every chunk, then the two components of
// the fields there.  As many buffers as fit: NB - 1 steps are in flight while one is computed.  A buffer also holds the
// transposed result of one component (chunks of at most 8 points).
template <int W>
struct Stage {
    static constexpr int P = 256 / W;  // most chunks of a block
    static constexpr int cols = W + 2, mat = 5 * cols, fld = 2 * cols;
    static constexpr int NB = W >= 4 ? 3 : 2;
    static constexpr int KM = (mat + 2 * W - 1) / (2 * W), KF = (fld + 2 * W - 1) / (2 * W);  // loads of a thread per step
    static constexpr int buffer = P * 2 * W * (KM + KF);
    static_assert(buffer >= W * (8 * P + P + 1) && NB * buffer * 16 <= 160 * 1024, "LDS of a block");
};

// waits until at most N of the wave's loads are in flight (and for its LDS reads), then for the block
template <int N>
__device__ __forceinline__ void wait_rows() {
    __builtin_amdgcn_s_waitcnt((N & 15) | (N >> 4) << 14 | 7 << 4);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// factors of the stencils, with the 1/4 of R and the dZ/2 of mu folded in
struct Steps {
    double l2, t2;    // d0: 1/dL^2, 1/dT^2
    double le, te;    // half of them (d1 takes the average of two 1/eps_zz)
    double c0;        // corners: 1 / (4 dL dT)
    double wl, wt;    // walk-off: 1 / (2 dL), 1 / (2 dT)
};

// what later rows need of a row
template <int NEU, int COMP>
struct Node {
    // tridiagonal row: along the line component d1 (a0 + ill_r a1) and walk-off a2 (u, kll, vl), along the transverse
    // one d0 (a0 + a0_r) + ilt_r d1 a1 (itt, klt)
    double e, a0, a1, a2;
    double ill, ilt, itt, ep, em, vt;
    // corner terms: differences over t, and the values at t + 1, t - 1
    c64 V, Q, Z, bp, bm, gp, gm;
    // Neumann launches: the own column's field component and material products on it
    c64 f;
    double m0, m1;
    c64 own;  // first launches: the right-hand side's part on this row
};

__device__ __forceinline__ c64 axby(double a, c64 x, double b, c64 y) {
    return mk(fma(a, x.x, b * y.x), fma(a, x.y, b * y.y));
}
__device__ __forceinline__ c64 madd(c64 acc, double a, c64 x) { return mk(fma(a, x.x, acc.x), fma(a, x.y, acc.y)); }
// a x + b y - (c z + d w)
__device__ __forceinline__ c64 diff2(double a, c64 x, double b, c64 y, double c, c64 z, double d, c64 w) {
    return madd(madd(axby(a, x, b, y), -c, z), -d, w);
}
// acc + i c - w
__device__ __forceinline__ c64 rot_add(c64 acc, c64 c, c64 w) { return mk(acc.x - c.y - w.x, acc.y + c.x - w.y); }

// mp, fl, ft: the row's material and fields in LDS at column t - 1
template <int NEU, int COMP>
__device__ __forceinline__ Node<NEU, COMP> make_node(const c64 *mp, const c64 *fl, const c64 *ft, const Steps &s) {
    using U = Uses<NEU, COMP>;
    Node<NEU, COMP> n;
    const Mat o = mat_of(mp + 5);
    n.e = o.e;
    n.ill = o.ill;
    n.ilt = o.ilt;
    n.itt = o.itt;
    n.vt = o.vt;
    if constexpr (COMP == 0) {
        n.a0 = fma(o.kll, o.ill, o.klt * o.ilt);
        n.a1 = o.kll;
        n.a2 = o.vl;
    } else {
        n.a0 = o.itt;
        n.a1 = o.klt;
    }
    c64 l0, t0;
    if constexpr (U::own_l) l0 = fl[1];
    if constexpr (U::own_t) t0 = ft[1];
    if constexpr (U::side) {
        const c64 ml = fl[0], mt = ft[0], pl = fl[2], pt = ft[2];
        const Mat m = mat_of(mp), p = mat_of(mp + 10);
        n.em = s.c0 * m.e;
        n.ep = s.c0 * p.e;
        const c64 dl = pl - ml, dt = pt - mt;
        // rows of K S^-1: (K S^-1)_tl, (K S^-1)_tt or _ll, _lt
        if constexpr (U::corner) {
            const double el = s.c0 * o.e;
            n.Z = dl;
            n.Q = axby(el, diff2(p.klt, pl, p.ktt, pt, m.klt, ml, m.ktt, mt), -s.c0, dt);
            n.bp = axby(p.kll, pl, p.klt, pt);
            n.bm = axby(m.kll, ml, m.klt, mt);
            if constexpr (NEU == 1) {
                const c64 dag = diff2(fma(p.klt, p.ill, p.ktt * p.ilt), pl, fma(p.klt, p.ilt, p.ktt * p.itt), pt,
                                      fma(m.klt, m.ill, m.ktt * m.ilt), ml, fma(m.klt, m.ilt, m.ktt * m.itt), mt);
                n.V = axby(el, dag, -s.c0, diff2(p.ilt, pl, p.itt, pt, m.ilt, ml, m.itt, mt));
            }
        }
        if constexpr (NEU == 0) {
            // stencils along t on this row: d0 with weights 1/dT^2, d1 with the averaged 1/eps_zz
            const double dm = s.te * (m.e + o.e), dp = s.te * (p.e + o.e);
            const c64 a0 = axby(o.klt, l0, o.ktt, t0);
            const c64 d1a = axby(dp, axby(p.klt, pl, p.ktt, pt) - a0, dm, axby(m.klt, ml, m.ktt, mt) - a0);
            const c64 d0l = (pl - l0) - (l0 - ml);
            if constexpr (COMP == 0) {
                const c64 g0 = axby(o.ill, l0, o.ilt, t0);
                const c64 d0g = (axby(p.ill, pl, p.ilt, pt) - g0) - (g0 - axby(m.ill, ml, m.ilt, mt));
                const c64 c = axby(s.t2, madd(d0g, o.ill, d0l), o.ilt, d1a);
                n.own = rot_add(l0, c, (s.wt * o.vl) * dt);
            } else {
                const c64 g0 = axby(fma(o.klt, o.ill, o.ktt * o.ilt), l0, fma(o.klt, o.ilt, o.ktt * o.itt), t0);
                const c64 gp = axby(fma(p.klt, p.ill, p.ktt * p.ilt), pl, fma(p.klt, p.ilt, p.ktt * p.itt), pt);
                const c64 gm = axby(fma(m.klt, m.ill, m.ktt * m.ilt), ml, fma(m.klt, m.ilt, m.ktt * m.itt), mt);
                const c64 c = madd(madd(axby(dp, gp - g0, dm, gm - g0), o.itt, d1a), s.t2 * o.ilt, d0l);
                const c64 wv = madd(madd(axby(p.vt + o.vt, pt, -(m.vt + o.vt), mt), p.vl, pl), -m.vl, ml);
                n.own = rot_add(t0, c, s.wt * wv);
                // corners: (K S^-1 f)_l at the two columns and the difference of (S^-1 f)_l
                n.V = diff2(p.ill, pl, p.ilt, pt, m.ill, ml, m.ilt, mt);
                n.gp = axby(fma(p.kll, p.ill, p.klt * p.ilt), pl, fma(p.kll, p.ilt, p.klt * p.itt), pt);
                n.gm = axby(fma(m.kll, m.ill, m.klt * m.ilt), ml, fma(m.kll, m.ilt, m.klt * m.itt), mt);
            }
        }
    }
    if constexpr (NEU == 1 && COMP == 0) {
        n.f = t0;
        n.m0 = fma(o.kll, o.ilt, o.klt * o.itt);
        n.m1 = o.klt;
    }
    if constexpr (NEU == 1 && COMP == 1) {
        n.f = l0;
        n.m1 = o.kll;
    }
    return n;
}

// what a row has gathered before its next neighbour is known
struct Carry {
    c64 part;       // right-hand side
    double cm;      // d1 weight towards the previous row
    double are, aim;
};

// corner terms of neighbour row q at row r
template <int NEU, int COMP>
__device__ __forceinline__ c64 corner(const Node<NEU, COMP> &r, const Node<NEU, COMP> &q, const Steps &s) {
    const c64 b = madd(axby(r.ep, q.bp, -r.em, q.bm), -s.c0, q.Z);
    if constexpr (NEU == 1) return madd(madd(q.V, r.ill, q.Q), r.ilt, b);
    else return madd(madd(madd(axby(r.ep, q.gp, -r.em, q.gm), -s.c0, q.V), r.itt, b), r.ilt, q.Q);
}

// Neumann coupling along the line of row r with its neighbour q over the edge of d1 weight ce (differences q - r):
// L_lt on the transverse component, L_tl on the line component
template <int NEU, int COMP>
__device__ __forceinline__ c64 along(double ce, const Node<NEU, COMP> &r, const Node<NEU, COMP> &q, const Steps &s) {
    if constexpr (COMP == 0) {
        const double d0 = r.ilt * s.l2;
        return axby(fma(ce, fma(r.ill, q.m1, q.m0), d0), q.f, -fma(ce, fma(r.ill, r.m1, r.m0), d0), r.f);
    } else {
        const double rc = r.ilt * ce;
        return axby(fma(s.l2, q.ilt, rc * q.m1), q.f, -fma(s.l2, r.ilt, rc * r.m1), r.f);
    }
}

// row r with its previous neighbour m
template <int NEU, int COMP>
__device__ __forceinline__ Carry begin_row(const Node<NEU, COMP> &m, const Node<NEU, COMP> &r, const Steps &s) {
    using U = Uses<NEU, COMP>;
    Carry k;
    k.cm = s.le * (m.e + r.e);
    if constexpr (COMP == 0) {
        k.are = k.cm * fma(r.ill, m.a1, m.a0);
        k.aim = -s.wl * (r.a2 + m.a2);
    } else {
        k.are = fma(s.l2, m.a0 + r.itt, r.ilt * k.cm * m.a1);
        k.aim = 0;
    }
    if constexpr (NEU == 1) {
        c64 c = along(k.cm, r, m, s);
        if constexpr (U::corner) c = c - corner(r, m, s);
        const double v = s.wl * (COMP == 0 ? m.vt : r.vt);
        k.part = mk(fma(v, m.f.x, -c.y), fma(v, m.f.y, c.x));
    } else {
        k.part = r.own;
        if constexpr (U::corner) {
            const c64 c = corner(r, m, s);
            k.part = mk(k.part.x + c.y, k.part.y - c.x);
        }
    }
    return k;
}

// the row (I - mu T) a, b, c and the right-hand side d of r, with its next neighbour p
template <int NEU, int COMP>
__device__ __forceinline__ void finish_row(const Carry &k, const Node<NEU, COMP> &r, const Node<NEU, COMP> &p,
                                           const Steps &s, c64 &a, c64 &b, c64 &cc, c64 &d) {
    using U = Uses<NEU, COMP>;
    const double cp = s.le * (p.e + r.e);
    a = mk(k.aim, -k.are);
    if constexpr (COMP == 0) {
        b = mk(1.0, (k.cm + cp) * fma(r.ill, r.a1, r.a0));
        cc = mk(s.wl * (r.a2 + p.a2), -cp * fma(r.ill, p.a1, p.a0));
    } else {
        b = mk(1.0, fma(4.0 * s.l2, r.itt, r.ilt * (k.cm + cp) * r.a1));
        cc = mk(0.0, -fma(s.l2, p.a0 + r.itt, r.ilt * cp * p.a1));
    }
    d = k.part;
    if constexpr (NEU == 1) {
        const c64 c = along(cp, r, p, s);
        const double v = s.wl * (COMP == 0 ? p.vt : r.vt);
        d = mk(fma(-v, p.f.x, d.x - c.y), fma(-v, p.f.y, d.y + c.x));
    }
    if constexpr (U::corner) {
        const c64 c = corner(r, p, s);
        d = mk(d.x - c.y, d.y + c.x);
    }
}

// a chunk of a line: interior rows 0 .. n-1 eliminated (responses to the right-hand side and to the last unknown of
// the chunk before; gam of row n-1 is the response to the chunk's own last unknown, with the sign turned), row n the
// interface
template <int STEPS>
struct WChunk {
    c64 gam[STEPS], yu[STEPS], yg[STEPS];
    c64 ul, gl, hl, uf, gf, hf;
    c64 ae, be, ce, de;
};

__device__ __forceinline__ void pick(bool take, c64 &to, c64 from) {
    to.x = take ? from.x : to.x;
    to.y = take ? from.y : to.y;
}

// f(I), ..., f(END - 1) of compile-time indices
template <int I, int END, class F>
__device__ __forceinline__ void static_for(F &&f) {
    if constexpr (I < END) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, END>(f);
    }
}

// The walk of one component's threads.  Both components' waves run it at once, each its own instance, and meet at the
// barriers of each step (a wave holds one component: P W is a multiple of 64).  Every row up to that of the longest
// chunk (STEPS) is computed by every thread; a chunk one row shorter takes its interface one row earlier.
template <int STEPS, int W, int NEU, int COMP, class Buf>
__device__ __forceinline__ void walk_lines(int tid, const LinePlan &lp, const c64 *mat, const c64 *fields,
                                           int line_comp, int tb, int Ml, int Mt, int NP, Buf &&rows, int p, int cc,
                                           bool is_short, const Steps &st, WChunk<STEPS> &ck) {
    using C = c64;
    using S = Stage<W>;
    typedef __attribute__((address_space(1))) const void *GPtr;
    typedef __attribute__((address_space(3))) void *LPtr;
    // Rows go straight to LDS, unit u of a step by lane u % 64 of load u / 64 (lanes past the last unit repeat it).  A
    // unit's chunk and column do not change: its byte offset at row 0 of the chunk is kept, the row comes with the
    // uniform base (the fields' base starts Ml rows before them, so that the offset of a row wrapped to the front stays
    // positive).  The material has the mesh's duplicate row and column as row Ml and column Mt, the fields are periodic.
    const int NT = lp.P * 2 * W, wave0 = __builtin_amdgcn_readfirstlane(tid & ~63);
    const unsigned ms = (unsigned)(Mt + 1) * 80, fs = (unsigned)Mt * 16;  // bytes of a row
    const int last_m = lp.P * S::mat, last_f = lp.P * S::fld;
    unsigned mo[S::KM], fo[S::KF];
#pragma unroll
    for (int k = 0; k < S::KM; k++) {
        const int u = min(tid + k * NT, last_m - 1), q = u / S::mat, off = u - q * S::mat, c = off / 5, col = tb - 1 + c;
        mo[k] = chunk_start(lp, q) * ms + (unsigned)(col < 0 ? Mt - 1 : min(col, Mt)) * 80 + (off - 5 * c) * 16;
    }
#pragma unroll
    for (int k = 0; k < S::KF; k++) {
        const int u = min(tid + k * NT, last_f - 1), q = u / S::fld, off = u - q * S::fld;
        const int comp = off < S::cols ? 0 : 1, col = tb - 1 + off - comp * S::cols;
        const int at = col < 0 ? Mt - 1 : col >= Mt ? min(col - Mt, Mt - 1) : col;
        fo[k] = (Ml + chunk_start(lp, q)) * fs + (unsigned)at * 16 +
                (comp == line_comp ? 0u : (unsigned)NP * 16);
    }
    auto fetch = [&](int j, c64 *buf) {  // rows j - 1 of the chunks
        const char *mb = reinterpret_cast<const char *>(mat) + (ptrdiff_t)(j - 1) * (ptrdiff_t)ms;
        const char *fb = reinterpret_cast<const char *>(fields) + (ptrdiff_t)(j - 1 - Ml) * (ptrdiff_t)fs;
#pragma unroll
        for (int k = 0; k < S::KM; k++) {
            const int u = tid + k * NT;
            unsigned o = mo[k];
            if (j == 0 && k == 0) o += u < S::mat ? Ml * ms : 0u;  // row -1 is row Ml - 1
            // a row past Ml (the last chunk is a row shorter): its values are not used
            if (j == STEPS + 1 && lp.rem) o -= u >= last_m - S::mat ? ms : 0u;
            __builtin_amdgcn_global_load_lds((GPtr)(mb + o), (LPtr)(buf + wave0 + k * NT), 16, 0, 0);
        }
#pragma unroll
        for (int k = 0; k < S::KF; k++) {
            const int u = tid + k * NT;
            unsigned o = fo[k];
            if (j == 0 && k == 0) o += u < S::fld ? Ml * fs : 0u;
            // rows Ml, Ml + 1 are rows 0, 1
            if (j > STEPS || (j == STEPS && lp.rem)) o -= u >= last_f - S::fld ? Ml * fs : 0u;
            __builtin_amdgcn_global_load_lds((GPtr)(fb + o), (LPtr)(buf + wave0 + (S::KM + k) * NT), 16, 0, 0);
        }
    };
    // rows(k) is buffer k, a static array of its own each: the compiler then knows that reading one does not wait for
    // the loads into another
    constexpr int NB = S::NB, LPS = S::KM + S::KF;
    static_assert(LPS * (NB - 2) < 64, "loads in flight");
    Node<NEU, COMP> cur;
    Carry kc;
    C binv{0, 0}, cprev{0, 0};
#pragma unroll
    for (int j = 0; j < NB - 1; j++)
        if (j < STEPS + 2) fetch(j, rows(j));
    static_for<0, STEPS + 2>([&](auto step) {
        constexpr int j = decltype(step)::value;
        // row j is in LDS once only the later rows' loads are in flight (near the end of the walk: none)
        wait_rows<j + NB - 2 < STEPS + 2 ? LPS * (NB - 2) : 0>();
        if constexpr (j + NB - 1 < STEPS + 2) fetch(j + NB - 1, rows((j + NB - 1) % NB));
        const c64 *mrow = rows(j % NB) + p * S::mat + 5 * cc, *frow = rows(j % NB) + S::KM * NT + p * S::fld + cc;
        const Node<NEU, COMP> nx = make_node<NEU, COMP>(mrow, frow, frow + S::cols, st);
        if constexpr (j == 1) kc = begin_row(cur, nx, st);
        if constexpr (j >= 2) {
            constexpr int i = j - 2;  // the row completed
            C a, b, c, d;
            finish_row<NEU, COMP>(kc, cur, nx, st, a, b, c, d);
            kc = begin_row(cur, nx, st);
            const C gm = cprev * binv;
            if constexpr (i > 0) ck.gam[i - 1] = gm;
            if constexpr (i >= STEPS - 2) {
                // the interface row: the last, or for short chunks the one before it
                const bool take = (i == STEPS - 1) != is_short;
                pick(take, ck.ae, a);
                pick(take, ck.be, b);
                pick(take, ck.ce, c);
                pick(take, ck.de, d);
                if constexpr (i > 0) {
                    pick(take, ck.ul, ck.yu[i - 1]);
                    pick(take, ck.gl, ck.yg[i - 1]);
                    pick(take, ck.hl, -gm);
                }
            }
            if constexpr (i == 0) {
                binv = wrcp(b);
                ck.yu[0] = d * binv;
                ck.yg[0] = -(a * binv);
            } else if constexpr (i + 1 < STEPS) {
                binv = wrcp(b - a * gm);
                ck.yu[i] = (d - a * ck.yu[i - 1]) * binv;
                ck.yg[i] = -(a * ck.yg[i - 1]) * binv;
            }
            cprev = c;
        }
        cur = nx;
        // a step at a time where the chains of longer chunks need the registers; else steps may overlap
        if constexpr (STEPS > 4) __builtin_amdgcn_sched_barrier(0);
    });
    // back substitution of the interior to its first unknown
    C u{0, 0}, g{0, 0}, h{1, 0};
#pragma unroll
    for (int i = STEPS - 2; i >= 0; i--) {
        const C nu = ck.yu[i] - ck.gam[i] * u, ng = ck.yg[i] - ck.gam[i] * g, nh = -(ck.gam[i] * h);
        const bool live = i < STEPS - 2 || !is_short;
        pick(live, u, nu);
        pick(live, g, ng);
        pick(live, h, nh);
    }
    ck.uf = u;
    ck.gf = g;
    ck.hf = h;
}

}  // namespace

// Lines along l: y = M_l (RHS of src), RHS (I + mu A_t) src (NEU 0) or mu O_l src (NEU 1); then dst = y and
// acc = accin + y (NEU 1) or y (NEU 0), a null dst or acc is skipped; with flip, acc is written in the order of
// the other axis ([t][l]).  axis 0: l = x, 1: l = y.  A block takes W adjacent lines of one propagation, both
// components, a thread one chunk of one component: 2 P W threads.  STEPS: rows of the longest chunk.
template <int STEPS, int W, int NEU>
__global__ __launch_bounds__(512) void k_walk(const c64 *__restrict__ src, c64 *__restrict__ dst,
                                              const c64 *accin, c64 *acc, WalkMaterial wm, int axis, int flip,
                                              Geo g, const PropParams *__restrict__ pp, LinePlan lp, int nprops,
                                              int per_slot) {
    using C = c64;
    using R = Stage<W>;
    // the rows; later the reduced systems, then the result
    __shared__ c64 rows0[R::buffer], rows1[R::buffer], rows2[R::NB > 2 ? R::buffer : 1];
    auto rows = [&](int k) { return k == 0 ? rows0 : k == 1 ? rows1 : rows2; };
    constexpr int lw = W == 16 ? 4 : W == 8 ? 3 : W == 4 ? 2 : 1;
    const int P = lp.P, TW = P * W, NT = 2 * TW;
    const int Ml = axis == 0 ? g.Mx : g.My, Mt = axis == 0 ? g.My : g.Mx;
    const int nstrip = (Mt + W - 1) / W;
    // work items: the propagations of one wavelength (they read the same material) innermost, then the strips, the
    // wavelengths outermost; every XCD takes a contiguous range
    const int item = xcd_tile(blockIdx.x, gridDim.x);
    if (item >= nstrip * nprops) return;
    const int group = item / (per_slot * nstrip), rest = item - group * per_slot * nstrip;
    const int strip = rest / per_slot, prop = group * per_slot + rest - strip * per_slot;
    const int tid = threadIdx.x;
    const int comp = __builtin_amdgcn_readfirstlane(tid >= TW ? 1 : 0);  // 0: the component along the line
    const int tl = tid - comp * TW;
    const int cc = tl & (W - 1), p = tl >> lw;
    const int tb = strip * W, t = tb + cc;
    const bool active = t < Mt;

    const int slot = pp[prop].slot;
    const WalkSteps &s = wm.steps[pp[prop].iwl];
    Steps st;
    st.l2 = axis == 0 ? s.rx2 : s.ry2;
    st.t2 = axis == 0 ? s.ry2 : s.rx2;
    st.le = 0.5 * st.l2;
    st.te = 0.5 * st.t2;
    st.c0 = s.rxy;
    st.wl = axis == 0 ? s.gx : s.gy;
    st.wt = axis == 0 ? s.gy : s.gx;

    const size_t NP = (size_t)g.NP, pb = (size_t)prop * 2 * NP;
    const c64 *mat = (axis == 0 ? wm.tr : wm.nat) + (size_t)slot * walk_points(g.Mx, g.My) * 5;

    const int s0 = chunk_start(lp, p), len = chunk_len(lp, p);
    WChunk<STEPS> ck;
    const bool is_short = len < STEPS;
    if (comp == 0)
        walk_lines<STEPS, W, NEU, 0>(tid, lp, mat, src + pb, axis, tb, Ml, Mt, (int)NP, rows, p, cc, is_short, st, ck);
    else
        walk_lines<STEPS, W, NEU, 1>(tid, lp, mat, src + pb, axis, tb, Ml, Mt, (int)NP, rows, p, cc, is_short, st, ck);
    __syncthreads();

    // the interface unknowns of the line's chunks: cyclic tridiagonal, A x_{p-1} + B x_p + C x_{p+1} = D, by cyclic
    // reduction with two LDS buffers of four arrays.  Each thread inverts its own B once a stage, for its neighbours.
    // The right-hand side is corrected, never rescaled: rows normalised to B = 1 take six values a stage (1024^2 x 200
    // 171.5 ms against 172.7, 512^2 x 100 17.2 against 17.3), but there the rounding of every stage reaches the unknowns
    // in full (error of the former 2.5e-15 against 5.7e-16, as the solvers on stored stencils).
    static_assert(4 * 2 * W * R::P <= R::buffer, "reduced systems");
    C *buf0 = rows0, *buf1 = rows1;
    buf0[tid] = ck.uf;
    buf0[NT + tid] = ck.gf;
    buf0[2 * NT + tid] = ck.hf;
    // the running sum is fetched while the reduction runs
    const size_t fo = pb + (size_t)(comp == (axis == 0 ? 0 : 1) ? 0 : 1) * NP + (active ? t : Mt - 1);
    C av[STEPS] = {};
    if (NEU && acc) {
#pragma unroll
        for (int i = 0; i < STEPS; i++)
            if (i + 1 < STEPS || !is_short) av[i] = accin[fo + (size_t)(s0 + i) * Mt];
    }
    __syncthreads();
    const int lb = comp * TW + cc;
    auto at = [&](int q) { return lb + ((q & (P - 1)) << lw); };
    C a, b, c, d;
    {
        const int nx = at(p + 1);
        const C ufn = buf0[nx], gfn = buf0[NT + nx], hfn = buf0[2 * NT + nx];
        a = ck.ae * ck.gl;
        b = ck.be + ck.ae * ck.hl + ck.ce * gfn;
        c = ck.ce * hfn;
        d = ck.de - ck.ae * ck.ul - ck.ce * ufn;
    }
    // to the other threads of the line: 1/B for a stage of the reduction, B for the last pairs
    auto publish = [&](C *x, C bv) {
        x[tid] = a;
        x[NT + tid] = bv;
        x[2 * NT + tid] = c;
        x[3 * NT + tid] = d;
        __syncthreads();
    };
    publish(buf1, wrcp(b));
    C *rd = buf1, *wr = buf0;
    for (int stp = 1; 2 * stp < P; stp <<= 1) {
        const int im = at(p - stp), iq = at(p + stp);
        const C k1 = a * rd[NT + im], k2 = c * rd[NT + iq];
        const C am = rd[im], cm = rd[2 * NT + im], dm = rd[3 * NT + im];
        const C aq = rd[iq], cq = rd[2 * NT + iq], dq = rd[3 * NT + iq];
        a = -(k1 * am);
        c = -(k2 * cq);
        b = b - k1 * cm - k2 * aq;
        d = d - k1 * dm - k2 * dq;
        publish(wr, 4 * stp < P ? wrcp(b) : b);
        C *x = rd;
        rd = wr;
        wr = x;
    }
    C xi;
    {
        const int q = at(p + P / 2);
        const C bq = rd[NT + q], dq = rd[3 * NT + q], b0 = a + c, b1 = rd[q] + rd[2 * NT + q];
        xi = (d * bq - b0 * dq) * wrcp(b * bq - b0 * b1);
    }
    wr[tid] = xi;
    __syncthreads();
    const C xprev = wr[at(p - 1)];

    // x_i = u_i + xprev g_i + xi h_i, last point first
    {
        C u{0, 0}, gg{0, 0}, h{1, 0};
#pragma unroll
        for (int i = STEPS - 1; i >= 0; i--) {
            if (i == STEPS - 1) {
                ck.yu[i] = xi;
                continue;
            }
            const bool live = i < STEPS - 2 || !is_short;  // (a short chunk's last point is this one)
            const C nu = ck.yu[i] - ck.gam[i] * u, ng = ck.yg[i] - ck.gam[i] * gg, nh = -(ck.gam[i] * h);
            pick(live, u, nu);
            pick(live, gg, ng);
            pick(live, h, nh);
            const C x = u + xprev * gg + xi * h;
            ck.yu[i] = x;
        }
    }
    if (dst && active) {
#pragma unroll
        for (int i = 0; i < STEPS; i++)
            if (i + 1 < STEPS || !is_short) dst[fo + (size_t)(s0 + i) * Mt] = ck.yu[i];
    }
    if (!acc) return;
#pragma unroll
    for (int i = 0; i < STEPS; i++)
        if (NEU) ck.yu[i] = av[i] + ck.yu[i];
    if (!flip) {
        if (active) {
#pragma unroll
            for (int i = 0; i < STEPS; i++)
                if (i + 1 < STEPS || !is_short) acc[fo + (size_t)(s0 + i) * Mt] = ck.yu[i];
        }
        return;
    }
    // the other axis' order, through LDS: line q of the block (component, line) is a run of Ml values, point l at
    // l + l / 8 so that the threads of a wave, eight points apart, fall on different banks
    const int ld = walk_line_pitch(Ml);
    __syncthreads();
    {
        C *row = (comp == 0 ? rows0 : rows1) + cc * ld;
#pragma unroll
        for (int i = 0; i < STEPS; i++)
            if (i + 1 < STEPS || !is_short) row[(s0 + i) + ((s0 + i) >> 3)] = ck.yu[i];
    }
    __syncthreads();
    const int lane = tid & 63, wave = tid >> 6, nwave = NT >> 6;
    for (int q = wave; q < 2 * W; q += nwave) {
        const int qc = q >> lw, to = tb + (q & (W - 1));
        if (to >= Mt) continue;
        C *o = acc + pb + (size_t)(qc == (axis == 0 ? 0 : 1) ? 0 : 1) * NP + (size_t)to * Ml;
        const C *row = (qc == 0 ? rows0 : rows1) + (q & (W - 1)) * ld;
        for (int l = lane; l < Ml; l += 64) o[l] = row[l + (l >> 3)];
    }
}

template <int W, int NEU>
static void walk_dispatch(const WalkShape &sh, dim3 grid, const c64 *src, c64 *dst, const c64 *accin, c64 *acc,
                          const WalkMaterial &wm, int axis, int flip, const Geo &g, const PropParams *pp,
                          int nprops, int per_slot, hipStream_t st) {
    const LinePlan &lp = sh.lp;
    const dim3 block(2 * lp.P * W);
    // two lines a block have 32 chunks or more, on lines of over 96 points: chunks of over 3
    const int steps = lp.base + (lp.rem ? 1 : 0);
    if (W == 2 && steps < 4) throw std::runtime_error("line walk: unsupported chunk length");
    switch (steps) {
#define NMK_STEPS(S)                                                                                                   \
    case S:                                                                                                            \
        if constexpr (W > 2 || S > 3)                                                                                  \
            hipLaunchKernelGGL((k_walk<S, W, NEU>), grid, block, 0, st, src, dst, accin, acc, wm, axis, flip, g, pp, \
                               lp, nprops, per_slot);                                                              \
        break;
        NMK_STEPS(2)
        NMK_STEPS(3)
        NMK_STEPS(4)
        NMK_STEPS(5)
        NMK_STEPS(6)
        NMK_STEPS(7)
        NMK_STEPS(8)
#undef NMK_STEPS
    default: throw std::runtime_error("line walk: unsupported chunk length");
    }
    NMK_WALK_CHECK();
}

void launch_walk(int axis, int neumann, const c64 *src, c64 *dst, const c64 *accin, c64 *acc, bool flip,
                 const WalkMaterial &wm, const Geo &g, const PropParams *pp, int nprops, int per_slot,
                 const WalkShape &sh, hipStream_t st) {
    const LinePlan &lp = sh.lp;
    const int Ml = axis == 0 ? g.Mx : g.My, Mt = axis == 0 ? g.My : g.Mx;
    // a wave holds chunks of one component; rows and result of a block fit its LDS buffers; the reduction takes a stage
    if (!g.px || !g.py || lp.M != Ml || lp.P < 4 || 2 * lp.P * sh.W > 512 ||
        lp.P * sh.W % 64 || per_slot < 1 || nprops % per_slot)
        throw std::runtime_error("line walk: bad launch shape");
    const int64_t items = (int64_t)((Mt + sh.W - 1) / sh.W) * nprops;
    if (items > 0x7ffffff8) throw std::runtime_error("line walk: too many work items");
    const dim3 grid((unsigned)((items + 7) / 8 * 8));
#define NMK_WALK(WW)                                                                                                    \
    if (sh.W == WW) {                                                                                                   \
        if (neumann) walk_dispatch<WW, 1>(sh, grid, src, dst, accin, acc, wm, axis, flip, g, pp, nprops, per_slot, st); \
        else walk_dispatch<WW, 0>(sh, grid, src, dst, accin, acc, wm, axis, flip, g, pp, nprops, per_slot, st);         \
        return;                                                                                                         \
    }
    NMK_WALK(16)
    NMK_WALK(8)
    NMK_WALK(4)
    NMK_WALK(2)
#undef NMK_WALK
    throw std::runtime_error("line walk: bad launch shape");
}

}  // namespace nmk
