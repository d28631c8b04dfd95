// C ABI of the engine: states, gates, observables, measurements and the
// adjoint Jacobian. See include/plk_amd.h for the contract of each entry
// point and the reference member it replaces.
#include <algorithm>
#include <type_traits>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <set>
#include <sstream>
#include <thread>
#include <tuple>

#include "plk_internal.hpp"

namespace plk {

namespace {

thread_local std::string g_last_error;

const cd kI{0.0, 1.0};

Device &dev_of(const State &s) { return device(s.device); }

// 64-bit structure hash (multiply-xorshift over 64-bit words).
struct Hasher {
    uint64_t h = 0x243F6A8885A308D3ull;
    void add(uint64_t v) {
        h ^= v + 0x9E3779B97F4A7C15ull + (h << 6) + (h >> 2);
        h *= 0xFF51AFD7ED558CCDull;
        h ^= h >> 32;
    }
    void add(double v) {
        uint64_t b;
        std::memcpy(&b, &v, sizeof b);
        add(b);
    }
    void add(const std::string &str) {
        add(static_cast<uint64_t>(str.size()));
        add(static_cast<uint64_t>(std::hash<std::string>{}(str)));
    }
};

// ---------------------------------------------------------------------------
// Observables (ObservablesKokkos.hpp:19-517).
// ---------------------------------------------------------------------------
struct ObsNode {
    enum Kind { Named, Hermitian, Tensor, Hamiltonian, Sparse } kind = Named;
    std::string name;
    std::vector<size_t> wires;
    std::vector<cd> matrix;
    std::vector<std::shared_ptr<const ObsNode>> terms;
    std::vector<double> coeffs;
    std::vector<double> data; // CSR values, interleaved complex
    std::vector<int64_t> indices, indptr;       // int64 matrices
    std::vector<int32_t> indices32, indptr32;   // int32 matrices (complex64 serialisation)
    bool idx32 = false;
    size_t rows = 0;
    // Hash of the tree (CSR values left out) without its matrices, whether it has
    // any, and the hash with them once a batched call has asked (see obs_key).
    uint64_t key = 0;
    bool dense = false;
    mutable uint64_t full_key = 0;
    mutable bool keyed = false;
    // Device copies of the CSR matrix per (device, state dtype), made on first
    // use and kept while the observable lives (entry points hold the engine
    // lock, so the cache needs no lock of its own).
    mutable std::map<std::pair<int, int>, std::unique_ptr<CsrDevice>> csr_dev;
    // Device Pauli tables per (device, qubit count) when the observable is a
    // sum of Pauli words (made on first use, kept while the observable lives).
    mutable std::map<std::pair<int, int>, std::unique_ptr<PauliDevice>> pauli_dev;
    const PauliDevice *pauli_on(Device &dev, int n) const;

    CsrView csr_view() const {
        CsrView v;
        v.data = data.data();
        v.idx32 = idx32;
        v.indices = idx32 ? static_cast<const void *>(indices32.data()) : indices.data();
        v.indptr = idx32 ? static_cast<const void *>(indptr32.data()) : indptr.data();
        v.nnz = data.size() / 2;
        v.rows = rows;
        return v;
    }
    const CsrDevice &csr_on(Device &dev, const State &s) const {
        auto &slot = csr_dev[{dev.id, s.dtype}];
        if (!slot) {
            const CsrView v = csr_view();
            csr_check_shape(v, s.len);
            slot = csr_upload(dev, v, s.dtype);
        }
        return *slot;
    }
};

// Hash of an observable's tree, for batched calls. All but the matrices is hashed
// with the observable (note_obs); hashing a matrix takes several times as long as
// copying it (10 wires: 2.8 ms to make the observable, 10.9 with the hash), so that
// is left to the first call that asks (under the engine lock).
uint64_t obs_key(const ObsNode &o) {
    if (!o.dense) {
        return o.key;
    }
    if (!o.keyed) {
        Hasher H;
        H.add(o.key);
        for (const cd &m : o.matrix) {
            H.add(m.real());
            H.add(m.imag());
        }
        for (const auto &t : o.terms) {
            H.add(obs_key(*t));
        }
        o.full_key = H.h;
        o.keyed = true;
    }
    return o.full_key;
}

void note_obs(ObsNode &o) {
    Hasher H;
    H.add(static_cast<uint64_t>(o.kind));
    H.add(o.name);
    H.add(static_cast<uint64_t>(o.wires.size()));
    for (auto w : o.wires) {
        H.add(static_cast<uint64_t>(w));
    }
    H.add(static_cast<uint64_t>(o.coeffs.size()));
    for (double c : o.coeffs) {
        H.add(c);
    }
    H.add(static_cast<uint64_t>(o.matrix.size()));
    H.add(static_cast<uint64_t>(o.terms.size()));
    o.dense = !o.matrix.empty();
    for (const auto &t : o.terms) {
        H.add(t->key);
        o.dense = o.dense || t->dense;
    }
    o.key = H.h;
}

std::vector<size_t> obs_wires(const ObsNode &o) {
    std::set<size_t> w;
    if (o.kind == ObsNode::Tensor || o.kind == ObsNode::Hamiltonian) {
        for (auto &t : o.terms) {
            auto tw = obs_wires(*t);
            w.insert(tw.begin(), tw.end());
        }
    } else {
        w.insert(o.wires.begin(), o.wires.end());
    }
    return {w.begin(), w.end()};
}

constexpr size_t kMaxPauliTerms = 4096;

uint64_t wire_bit(int n, size_t w) {
    if (w >= static_cast<size_t>(n)) {
        raise(PLK_ERR_INVALID, "observable wire " + std::to_string(w) + " out of range");
    }
    return uint64_t{1} << (n - 1 - static_cast<int>(w));
}

// Expands an observable into Pauli words when it is a sum of products of
// Identity / PauliX / PauliY / PauliZ / Hadamard with at most cap words.
// Returns false otherwise.
bool to_pauli(const ObsNode &o, int n, std::vector<PauliTerm> &out,
              size_t cap = kMaxPauliTerms) {
    switch (o.kind) {
    case ObsNode::Named: {
        if (o.name == "Identity") {
            out = {PauliTerm{0, 0, 1.0}};
            return true;
        }
        if (o.wires.size() != 1) {
            return false;
        }
        const uint64_t b = wire_bit(n, o.wires[0]);
        if (o.name == "PauliX") {
            out = {PauliTerm{b, 0, 1.0}};
        } else if (o.name == "PauliY") {
            out = {PauliTerm{b, b, -kI}};
        } else if (o.name == "PauliZ") {
            out = {PauliTerm{0, b, 1.0}};
        } else if (o.name == "Hadamard") {
            out = {PauliTerm{b, 0, M_SQRT1_2}, PauliTerm{0, b, M_SQRT1_2}};
        } else {
            return false;
        }
        return true;
    }
    case ObsNode::Tensor: {
        std::vector<PauliTerm> acc{PauliTerm{0, 0, 1.0}};
        for (auto &f : o.terms) {
            std::vector<PauliTerm> ft;
            if (!to_pauli(*f, n, ft, cap)) {
                return false;
            }
            std::vector<PauliTerm> next;
            if (acc.size() * ft.size() > cap) {
                return false;
            }
            for (auto &a : acc) {
                for (auto &b : ft) {
                    // Factors act on disjoint wires, so words multiply bitwise.
                    next.push_back({a.x | b.x, a.zy | b.zy, a.coeff * b.coeff});
                }
            }
            acc.swap(next);
        }
        out = acc;
        return true;
    }
    case ObsNode::Hamiltonian: {
        std::vector<PauliTerm> acc;
        for (size_t t = 0; t < o.terms.size(); t++) {
            std::vector<PauliTerm> tt;
            if (!to_pauli(*o.terms[t], n, tt, cap)) {
                return false;
            }
            for (auto &p : tt) {
                p.coeff *= o.coeffs[t];
                acc.push_back(p);
            }
            if (acc.size() > cap) {
                return false;
            }
        }
        out = acc;
        return true;
    }
    default:
        return false;
    }
}

// ---------------------------------------------------------------------------
// Gate application.
// ---------------------------------------------------------------------------
// A trainable gate of a fused run: its Jacobian column and coefficient, and
// the operator V^dag G V (V the run's gates before it) as m0 X + m1 Y + m2 Z.
struct RunTerm {
    int col;
    double coef;
    double m[3];
};

// A gate of a run in a batch plan: its patch, or the matrix it always has.
struct RunGate {
    BatchGate g{};
    std::vector<cd> mat; // BPG_CONST
};

struct PlanOp {
    CompiledOp U;
    std::vector<RunGate> gates; // batch plans: the gates of a one-wire op, in order
    std::vector<RunTerm> run; // register-tile plans: the trainable gates of a one-wire run
    bool trainable = false;
    CompiledGen G;
    int col = -1;
    double coef = 0.0;
    int32_t src = -1;       // index of the op in its OpsData
    bool adj = false;       // U was compiled with the inverse flag set
    bool skew = false;      // reverse sweeps: U is not unitary, or may not be (see Blocked)
    uint64_t mix = 0;       // register-tile plans: the state bits it mixes
    // Batch plans, runs with patched gates: the U kind and the Pauli parts that
    // hold for every angle (see fix_form); -1: as the matrices are.
    int ukind = -1, parts = -1;
};

// Parity ops/generators on <= 2 wires become dense diagonals so they fuse.
std::vector<cd> parity_diag(size_t m, cd even, cd odd) {
    const size_t dim = size_t{1} << m;
    std::vector<cd> M(dim * dim, 0.0);
    for (size_t r = 0; r < dim; r++) {
        M[r * dim + r] = (__builtin_popcountll(r) & 1) ? odd : even;
    }
    return M;
}

void densify(CompiledOp &op) {
    if (op.kind == OpKind::Parity && op.wires.size() <= 2) {
        op.mat = parity_diag(op.wires.size(), op.even, op.odd);
        op.kind = OpKind::Dense;
    }
}

void densify(CompiledGen &g) {
    if (g.kind == OpKind::Parity && g.wires.size() <= 2) {
        g.mat = parity_diag(g.wires.size(), 1.0, -1.0);
        g.kind = OpKind::Dense;
    }
}

bool fusable(const PlanOp &p) {
    if (p.U.kind != OpKind::Dense || p.U.wires.size() > 2) {
        return false;
    }
    if (p.trainable && (p.G.kind != OpKind::Dense || p.G.wires.size() > 2)) {
        return false;
    }
    return true;
}

struct Segment {
    std::vector<size_t> wires; // global wires of the segment
    std::vector<PlanOp> ops;
    int nslots = 0;
};

// A tile pass: bundles of ops on at most two tile bits each, all inside the
// pass's T tile bits.
struct Bundle {
    int K = 1;
    int qa = 0, qb = 0; // tile-local positions, qa > qb when K == 2
    std::vector<PlanOp> ops;
    int nslots = 0;
};

struct Pass {
    std::vector<int> tb; // ascending global bit positions
    std::vector<Bundle> bundles;
    std::vector<PlanOp> ops; // register-tile passes: the ops in program order
    bool rt = false;         // a register-tile pass (ops) rather than LDS bundles
    int nslots = 0;            // sums (LDS passes: one per trainable op)
    std::vector<int> cols;     // Jacobian column of each trainable op, in order
    std::vector<double> coefs; // and its coefficient
};

struct Step {
    bool fused = false; // register segment
    bool tiled = false; // LDS tile pass
    Segment seg;
    Pass pass;
    PlanOp single;
};

constexpr size_t kSegMaxOps = 64;

// Greedy fusion of consecutive operations into register segments.
std::vector<Step> plan_steps(std::vector<PlanOp> &&ops) {
    std::vector<Step> steps;
    Segment cur;
    auto flush = [&]() {
        if (!cur.ops.empty()) {
            Step s;
            s.fused = true;
            s.seg = std::move(cur);
            steps.push_back(std::move(s));
        }
        cur = Segment{};
    };
    for (auto &p : ops) {
        if (p.U.kind == OpKind::Identity && !p.trainable) {
            continue;
        }
        densify(p.U);
        if (p.trainable) {
            densify(p.G);
        }
        if (!fusable(p)) {
            flush();
            Step s;
            s.fused = false;
            s.single = std::move(p);
            steps.push_back(std::move(s));
            continue;
        }
        std::set<size_t> w(cur.wires.begin(), cur.wires.end());
        w.insert(p.U.wires.begin(), p.U.wires.end());
        if (w.size() > static_cast<size_t>(SEG_KMAX) || cur.ops.size() >= kSegMaxOps ||
            (p.trainable && cur.nslots >= SEG_PMAX)) {
            flush();
            w = std::set<size_t>(p.U.wires.begin(), p.U.wires.end());
        }
        cur.wires.assign(w.begin(), w.end());
        if (p.trainable) {
            cur.nslots++;
        }
        cur.ops.push_back(std::move(p));
    }
    flush();
    return steps;
}

void prepare(PlanOp &p) {
    densify(p.U);
    if (p.trainable) {
        densify(p.G);
    }
}

constexpr size_t kPassMaxOps = 512;
constexpr size_t kBundleLookahead = 64;
constexpr size_t kLookahead = 512;

// Splits a pass's ops (in order) into bundles of <= 2 tile bits.
void make_bundles(Pass &ps, std::vector<PlanOp> &&ops, int n) {
    int pos[64];
    for (size_t q = 0; q < ps.tb.size(); q++) {
        pos[ps.tb[q]] = static_cast<int>(q);
    }
    std::vector<PlanOp> all = std::move(ops);
    std::vector<uint32_t> obits(all.size());
    std::vector<uint64_t> wmask(all.size());
    std::vector<int> rem(all.size());
    for (size_t i = 0; i < all.size(); i++) {
        uint32_t ob = 0;
        uint64_t wm = all[i].skew ? ~uint64_t{0} : 0;
        for (auto w : all[i].U.wires) {
            ob |= 1u << pos[n - 1 - static_cast<int>(w)];
            wm |= uint64_t{1} << w;
        }
        obits[i] = ob;
        wmask[i] = wm;
        rem[i] = static_cast<int>(i);
    }
    // Each bundle starts at the first remaining op and takes later ops that
    // fit its two tile bits, provided no skipped op before them shares a
    // wire (ops on disjoint wires commute), within a window of kBundleLookahead.
    std::vector<int> rest;
    while (!rem.empty()) {
        Bundle cur;
        uint32_t cb = 0;
        uint64_t blocked = 0;
        rest.clear();
        size_t k = 0;
        for (; k < rem.size() && k < kBundleLookahead; k++) {
            const int i = rem[k];
            PlanOp &p = all[i];
            const bool ok = !(blocked & wmask[i]) && __builtin_popcount(cb | obits[i]) <= 2 &&
                            cur.ops.size() < kSegMaxOps && (!p.trainable || cur.nslots < SEG_PMAX);
            if (ok) {
                cb |= obits[i];
                if (p.trainable) {
                    cur.nslots++;
                    ps.cols.push_back(p.col);
                    ps.coefs.push_back(p.coef);
                    ps.nslots++;
                }
                cur.ops.push_back(std::move(p));
            } else {
                blocked |= wmask[i];
                rest.push_back(i);
            }
        }
        rest.insert(rest.end(), rem.begin() + static_cast<long>(k), rem.end());
        const int lo = __builtin_ctz(cb);
        if (__builtin_popcount(cb) == 1) {
            cur.K = 1;
            cur.qa = lo;
        } else {
            cur.K = 2;
            cur.qa = 31 - __builtin_clz(cb);
            cur.qb = lo;
        }
        ps.bundles.push_back(std::move(cur));
        rem.swap(rest);
    }
}

// True when the dim x dim matrix M has a nonzero entry between local
// indices that differ in local bit lb.
bool mixes_bit(const std::vector<cd> &M, int dim, int lb) {
    for (int r = 0; r < dim; r++) {
        for (int c = 0; c < dim; c++) {
            if ((((r ^ c) >> lb) & 1) && M[static_cast<size_t>(r) * dim + c] != cd(0.0, 0.0)) {
                return true;
            }
        }
    }
    return false;
}

// Pauli parts the gates of a run need: bit 0 X, bit 1 Y, bit 2 Z.
int run_parts(const PlanOp &p) {
    if (p.parts >= 0) {
        return p.parts;
    }
    int parts = 0;
    for (const auto &t : p.run) {
        for (int k = 0; k < 3; k++) {
            parts |= t.m[k] != 0.0 ? 1 << k : 0;
        }
    }
    return parts;
}

// Sums a register-tile pass keeps for an op.
int rt_slots(const PlanOp &p) {
    if (p.run.empty()) {
        return p.trainable ? 1 : 0;
    }
    const int parts = run_parts(p);
    return (parts & (parts - 1)) ? 3 : 1;
}

// 2x2 product A B.
std::vector<cd> mul2(const std::vector<cd> &A, const std::vector<cd> &B) {
    return {A[0] * B[0] + A[1] * B[2], A[0] * B[1] + A[1] * B[3], A[2] * B[0] + A[3] * B[2],
            A[2] * B[1] + A[3] * B[3]};
}

// Fuses the one-wire ops that follow each other on a wire into one 2x2
// matrix, at the place of the first (ops on other wires commute with them).
// Trainable ops join when their generator is traceless (X, Y, Z and real
// combinations of them); anything else on the wire ends the run. A skew op of a
// reverse sweep ends every run, and no trainable op joins the one it begins
// (V^dag G V would have a trace).
std::vector<PlanOp> fuse_runs(std::vector<PlanOp> &&ops) {
    std::vector<PlanOp> out;
    out.reserve(ops.size());
    std::vector<long> open(64, -1);
    for (auto &p : ops) {
        if (p.U.kind == OpKind::Identity && !p.trainable) {
            continue;
        }
        prepare(p);
        bool one = p.U.kind == OpKind::Dense && p.U.wires.size() == 1;
        if (one && p.trainable) {
            one = p.G.kind == OpKind::Dense && p.G.wires == p.U.wires && p.G.mat[0] + p.G.mat[3] == cd(0.0, 0.0);
        }
        if (!one) {
            if (p.skew) {
                std::fill(open.begin(), open.end(), -1);
            }
            for (auto w : p.U.wires) {
                open[w] = -1;
            }
            out.push_back(std::move(p));
            continue;
        }
        const size_t w = p.U.wires[0];
        if (p.skew) {
            std::fill(open.begin(), open.end(), -1);
        }
        const bool first = open[w] < 0 || (p.trainable && out[open[w]].skew);
        if (p.trainable) {
            std::vector<cd> g = p.G.mat;
            if (!first) {
                const std::vector<cd> &V = out[open[w]].U.mat;
                const std::vector<cd> Vd = {std::conj(V[0]), std::conj(V[2]), std::conj(V[1]), std::conj(V[3])};
                g = mul2(Vd, mul2(g, V));
            }
            const RunTerm t{p.col, p.coef,
                            {0.5 * (g[1] + g[2]).real(), 0.5 * (g[2].imag() - g[1].imag()),
                             0.5 * (g[0] - g[3]).real()}};
            PlanOp &into = first ? p : out[open[w]];
            into.run.push_back(t);
            into.trainable = true;
        }
        if (first) {
            open[w] = static_cast<long>(out.size());
            out.push_back(std::move(p));
        } else {
            PlanOp &o = out[open[w]];
            o.gates.insert(o.gates.end(), p.gates.begin(), p.gates.end());
            o.U.mat = mul2(p.U.mat, o.U.mat);
        }
    }
    return out;
}

// Whether a gate of a batch run is diagonal, whether it is real, and for each
// Pauli P (X, Y, Z) the parts that M^dag P M may have, M the gate's matrix at
// any angle.
struct GateForm {
    bool diag, real;
    int reach[3];
};

GateForm gate_form(const RunGate &g) {
    switch (g.g.gate) {
    case BPG_RX:
        return {false, false, {1, 6, 6}};
    case BPG_RY:
        return {false, true, {5, 2, 5}};
    case BPG_RZ:
    case BPG_PHASE:
        return {true, false, {3, 3, 4}};
    default:
        break;
    }
    const std::vector<cd> &M = g.mat;
    const std::vector<cd> Md = {std::conj(M[0]), std::conj(M[2]), std::conj(M[1]), std::conj(M[3])};
    const std::vector<cd> P[3] = {{0.0, 1.0, 1.0, 0.0}, {0.0, -kI, kI, 0.0}, {1.0, 0.0, 0.0, -1.0}};
    const cd none(0.0, 0.0);
    GateForm f{M[1] == none && M[2] == none, true, {0, 0, 0}};
    for (const cd &m : M) {
        f.real = f.real && m.imag() == 0.0;
    }
    for (int k = 0; k < 3; k++) {
        const std::vector<cd> W = mul2(Md, mul2(P[k], M));
        f.reach[k] = (W[1] + W[2] != none ? 1 : 0) | (W[1] != W[2] ? 2 : 0) | (W[0] != W[3] ? 4 : 0);
    }
    return f;
}

// The kind of a batch run's matrix and its Pauli parts, from the kinds of its
// gates. A plan serves every angle of its patched gates, so neither may come
// from the product at some angles: RX(a) Z RX(b) is diagonal at a = b only, and
// RY(a) RY(b)^dag the identity.
void fix_form(PlanOp &p) {
    bool patched = false;
    for (const RunGate &g : p.gates) {
        patched = patched || g.g.gate != BPG_CONST;
    }
    if (!patched) {
        return;
    }
    bool diag = true, real = true;
    int parts = 0;
    int reach[3] = {1, 2, 4}; // of V^dag P V, V the gates so far
    for (const RunGate &g : p.gates) {
        const GateForm f = gate_form(g);
        if (g.g.coef != 0.0) { // its generator: X, Y, else Z
            parts |= reach[g.g.gate == BPG_RX ? 0 : g.g.gate == BPG_RY ? 1 : 2];
        }
        int next[3] = {0, 0, 0};
        for (int k = 0; k < 3; k++) {
            for (int q = 0; q < 3; q++) {
                next[k] |= (f.reach[k] >> q & 1) ? reach[q] : 0;
            }
        }
        std::copy(next, next + 3, reach);
        diag = diag && f.diag;
        real = real && f.real;
    }
    p.ukind = diag ? U_DIAG : real ? U_REAL : U_DENSE;
    p.parts = p.run.empty() ? -1 : parts;
}

// Global state bits an op mixes (its U or, when trainable, its generator has
// an entry between indices that differ in the bit).
uint64_t mixing_mask(const PlanOp &p, int n) {
    const int m = static_cast<int>(p.U.wires.size());
    uint64_t mask = 0;
    if (!p.run.empty() || p.ukind >= 0) {
        const bool mixes = (p.ukind >= 0 ? p.ukind != U_DIAG : mixes_bit(p.U.mat, 2, 0)) ||
                           (!p.run.empty() && run_parts(p) != 4);
        return mixes ? uint64_t{1} << (n - 1 - static_cast<int>(p.U.wires[0])) : 0;
    }
    for (int k = 0; k < m; k++) {
        const int lb = m - 1 - k;
        if (mixes_bit(p.U.mat, 1 << m, lb) || (p.trainable && mixes_bit(p.G.mat, 1 << m, lb))) {
            mask |= uint64_t{1} << (n - 1 - static_cast<int>(p.U.wires[k]));
        }
    }
    return mask;
}

// The state bits an operation acts on and those it mixes; whether it leaves a
// derivative, and whether it is a matrix that is not unitary.
struct Place {
    uint64_t on = 0, mix = 0;
    bool trainable = false, skew = false;
};

// Operations skipped so far: the bits they mix, and the bits they act on,
// which stop an operation that mixes them. Operations that share only bits
// neither mixes commute. A trainable and a skew operation never change places:
// the derivative Im<h|G phi> is the same before and after a unitary on other
// wires, but not a matrix A, which makes it Im<h|A^dag A G phi>.
struct Blocked {
    uint64_t mixed = 0, selected = 0;
    bool trainable = false, skew = false;
    bool stops(const Place &p) const {
        return ((mixed & p.on) | (selected & p.mix)) != 0 || (trainable && p.skew) || (skew && p.trainable);
    }
    void add(const Place &p) {
        mixed |= p.mix;
        selected |= p.on;
        trainable = trainable || p.trainable;
        skew = skew || p.skew;
    }
};

// Groups operations into LDS tile passes of T bits that always contain the
// lowest L bits. Operations on disjoint wires commute, so an operation may be
// taken ahead of skipped ones it shares no wire with; an unfusable operation
// is a barrier and runs on its own. With bundled == false (register-tile
// passes) one-wire runs are fused first, a pass needs in its tile only the
// bits its operations mix, and operations that share only wires which neither
// mixes commute as well.
//
// A pass's tile starts as the bits of the first operations that fit. With
// `exchange` each of them is then exchanged for the outside bit with which the
// pass takes most operations, if any takes more. A trial walks the operations
// until every wire is blocked.
std::vector<Step> plan_tiles(std::vector<PlanOp> &&ops_in, int n, int T, int L,
                             int pmax = TILE_PMAX, bool bundled = true, bool exchange = false) {
    std::vector<PlanOp> all;
    if (bundled) {
        for (auto &p : ops_in) {
            if (p.U.kind == OpKind::Identity && !p.trainable) {
                continue;
            }
            prepare(p);
            all.push_back(std::move(p));
        }
    } else {
        all = fuse_runs(std::move(ops_in));
        for (PlanOp &p : all) {
            fix_form(p);
        }
    }
    // State bits (< 64) an op acts on, and of these the ones its pass needs in
    // the tile.
    struct Item : Place {
        int index, sums;
        bool fus;
    };
    std::vector<Item> items(all.size());
    uint64_t every = 0;
    for (size_t i = 0; i < all.size(); i++) {
        Item &it = items[i];
        it.index = static_cast<int>(i);
        it.trainable = all[i].trainable;
        it.skew = all[i].skew;
        for (auto w : all[i].U.wires) {
            it.on |= uint64_t{1} << (n - 1 - static_cast<int>(w));
        }
        every |= it.on;
        it.fus = fusable(all[i]);
        it.mix = bundled || !it.fus ? it.on : mixing_mask(all[i], n);
        all[i].mix = it.mix;
        it.sums = bundled ? (all[i].trainable ? 1 : 0) : rt_slots(all[i]);
    }
    // The first kLookahead operations left, all that a pass looks at: those that
    // earlier passes skipped, then items from `next` on.
    std::vector<Item> rem, rest;
    size_t next = 0;
    auto refill = [&] {
        const size_t add = std::min(kLookahead - rem.size(), items.size() - next);
        rem.insert(rem.end(), items.begin() + static_cast<long>(next), items.begin() + static_cast<long>(next + add));
        next += add;
    };
    // Operations of rem that a pass over these bits takes.
    auto count = [&](uint64_t bits) {
        Blocked blocked;
        size_t taken = 0;
        int sums = 0;
        for (size_t k = 0; k < rem.size() && rem[k].fus && (blocked.mixed & every) != every; k++) {
            const Item &it = rem[k];
            if ((it.mix & ~bits) == 0 && !blocked.stops(it) && taken < kPassMaxOps && sums + it.sums <= pmax) {
                taken++;
                sums += it.sums;
            } else {
                blocked.add(it);
            }
        }
        return taken;
    };
    const uint64_t low = L > 0 ? (uint64_t{1} << L) - 1 : 0;
    std::vector<Step> steps;
    std::vector<int> taken;
    for (refill(); !rem.empty(); refill()) {
        if (!rem[0].fus) {
            Step s;
            s.single = std::move(all[rem[0].index]);
            steps.push_back(std::move(s));
            rem.erase(rem.begin());
            continue;
        }
        // Bits of the first operations that fit, then the lowest unused ones.
        uint64_t bits = low;
        auto pad = [&] {
            for (int b = 0; __builtin_popcountll(bits) < T && b < n; b++) {
                bits |= uint64_t{1} << b;
            }
        };
        int nslots = 0;
        auto take = [&](bool grow) {
            Blocked blocked;
            taken.clear();
            rest.clear();
            nslots = 0;
            size_t k = 0;
            for (; k < rem.size() && rem[k].fus; k++) {
                const Item &it = rem[k];
                const uint64_t nb = bits | it.mix;
                if ((grow ? __builtin_popcountll(nb) <= T : nb == bits) && !blocked.stops(it) &&
                    taken.size() < kPassMaxOps && nslots + it.sums <= pmax) {
                    bits = nb;
                    nslots += it.sums;
                    taken.push_back(it.index);
                } else {
                    blocked.add(it);
                    rest.push_back(it);
                }
            }
            rest.insert(rest.end(), rem.begin() + static_cast<long>(k), rem.end());
        };
        take(true);
        pad();
        if (exchange && !rest.empty() && rest[0].fus) {
            const uint64_t before = bits;
            size_t best = count(bits);
            for (uint64_t outs = bits & ~low; outs != 0; outs &= outs - 1) {
                const uint64_t others = bits & ~(outs & (~outs + 1));
                for (uint64_t ins = every & ~bits; ins != 0; ins &= ins - 1) {
                    const uint64_t trial = others | (ins & (~ins + 1));
                    const size_t c = count(trial);
                    if (c > best) {
                        best = c;
                        bits = trial;
                    }
                }
            }
            if (bits != before || best > taken.size()) {
                take(false);
            }
        }
        Step s;
        s.tiled = true;
        for (int b = 0; b < 64; b++) {
            if (bits >> b & 1) {
                s.pass.tb.push_back(b);
            }
        }
        std::vector<PlanOp> ops;
        ops.reserve(taken.size());
        for (int i : taken) {
            ops.push_back(std::move(all[i]));
        }
        if (bundled) {
            make_bundles(s.pass, std::move(ops), n);
        } else {
            s.pass.nslots = nslots;
            s.pass.ops = std::move(ops);
            s.pass.rt = true;
        }
        steps.push_back(std::move(s));
        rem.swap(rest);
    }
    return steps;
}

int low_bits(int dtype) { return dtype == PLK_C64 ? 4 : 3; }

int env_int(const char *name, int dflt) {
    const char *v = std::getenv(name);
    return v && *v ? std::atoi(v) : dflt;
}

// Whether a register-tile plan for this many states exchanges tile bits: the
// trials take 20 to 30 us of host time a pass and save a fifth to a quarter of
// the passes, which pays from 1 GiB moved a pass on (25-qubit complex128 gate
// stream, 1 GiB: 6.3 ms without and 5.6 with; 24 qubits 2.67 and 2.84; 24-qubit
// complex128 Jacobian of 9 observables, 5 GiB: 37 passes and 60.4 ms without,
// 29 and 54.3 with).
bool plan_exchange(int n, int dtype, size_t states) {
    return 2.0 * static_cast<double>(states) * std::ldexp(dtype == PLK_C64 ? 8.0 : 16.0, n) >= 1073741824.0;
}

// Tile width of backward (adjoint) passes; 0 selects register segments.
int tile_bits_adjoint(int n, int dtype) {
    if (env_int("PLK_TILES", 1) == 0) {
        return 0;
    }
    const int T = std::min({env_int("PLK_TILE_BITS_ADJ", 10), n - 8, TILE_TMAX});
    return T >= low_bits(dtype) + 2 ? T : 0;
}

int tile_bits_forward(int n, int dtype) {
    if (env_int("PLK_TILES", 1) == 0) {
        return 0;
    }
    const int T = std::min({env_int("PLK_TILE_BITS_FWD", dtype == PLK_C64 ? 11 : 10), n - 8, TILE_TMAX});
    return T >= low_bits(dtype) + 2 ? T : 0;
}

// Largest observable chunk whose tiles fit the LDS budget.
int tile_max_nj(int dtype, int T) {
    int best = 1;
    const int cap = env_int("PLK_TILE_NJ", 4);
    for (int nj = 1; nj <= 8; nj++) {
        if (tile_nj_supported(dtype, nj) &&
            tile_lds_bytes(dtype, T, nj, TILE_PMAX) <= TILE_LDS_MAX && nj <= cap) {
            best = nj;
        }
    }
    return best;
}

// n_obs split into balanced chunks of at most njmax.
std::vector<int> chunk_sizes(size_t n_obs, int njmax) {
    const size_t k = (n_obs + njmax - 1) / njmax;
    std::vector<int> out;
    for (size_t c = 0; c < k; c++) {
        out.push_back(static_cast<int>(n_obs / k + (c < n_obs % k ? 1 : 0)));
    }
    return out;
}

struct SegMeta {
    SegLaunch L{};
    size_t first = 0; // byte offset of the segment's op group in the table
    int cols[SEG_PMAX] = {0};
    double coefs[SEG_PMAX] = {0};
    TileLaunch TL{};
    size_t first_bundle = 0;
};

template <typename T>
void put_mat(T *dst, const std::vector<cd> &M, bool swap_bits) {
    const size_t dim = M.size() == 16 ? 4 : 2;
    auto sw = [&](size_t r) { return swap_bits ? (((r & 1) << 1) | ((r >> 1) & 1)) : r; };
    for (size_t r = 0; r < dim; r++) {
        for (size_t c = 0; c < dim; c++) {
            const cd v = M[sw(r) * dim + sw(c)];
            dst[2 * (r * dim + c)] = static_cast<T>(v.real());
            dst[2 * (r * dim + c) + 1] = static_cast<T>(v.imag());
        }
    }
}

template <typename T>
size_t pack_ops(std::vector<unsigned char> &out, const SegOp<T> *ops, size_t nops) {
    auto align16 = [&]() { out.resize((out.size() + 15) & ~size_t{15}, 0); };
    align16();
    const size_t base = out.size();
    out.resize(base + nops * sizeof(OpHead), 0);
    for (size_t o = 0; o < nops; o++) {
        const SegOp<T> &d = ops[o];
        const int dim = d.m == 1 ? 2 : 4;
        T u[32], g[32];
        int nu = 0, ng = 0;
        switch (d.ukind) {
        case U_DIAG:
            for (int r = 0; r < dim; r++) {
                u[nu++] = d.U[2 * (r * dim + r)];
                u[nu++] = d.U[2 * (r * dim + r) + 1];
            }
            break;
        case U_REAL:
            for (int e = 0; e < dim * dim; e++) {
                u[nu++] = d.U[2 * e];
            }
            break;
        case U_SWAP:
            break;
        default:
            for (int e = 0; e < 2 * dim * dim; e++) {
                u[nu++] = d.U[e];
            }
        }
        if (d.slot >= 0) {
            if (d.gkind == G_DIAG) {
                for (int r = 0; r < dim; r++) {
                    g[ng++] = d.G[2 * (r * dim + r)];
                }
            } else if (d.gkind == G_DENSE) {
                for (int e = 0; e < 2 * dim * dim; e++) {
                    g[ng++] = d.G[e];
                }
            }
        }
        align16();
        const size_t uoff = out.size() - base;
        out.insert(out.end(), reinterpret_cast<const unsigned char *>(u),
                   reinterpret_cast<const unsigned char *>(u + nu));
        align16();
        const size_t goff = out.size() - base;
        out.insert(out.end(), reinterpret_cast<const unsigned char *>(g),
                   reinterpret_cast<const unsigned char *>(g + ng));
        if (goff > 0xffff) {
            raise(PLK_ERR_UNSUPPORTED, "operation group exceeds 64 KiB");
        }
        OpHead h{};
        h.cls = d.cls;
        h.slot = d.slot;
        h.kinds = d.ukind | (d.gkind << 8) | (d.swap << 16);
        h.offs = static_cast<int32_t>(uoff | (goff << 16));
        std::memcpy(out.data() + base + o * sizeof(OpHead), &h, sizeof(OpHead));
    }
    align16();
    return base;
}

// Picks the structure-specialized kernel path for a descriptor whose U (and
// G) already hold the final, bit-permuted matrices of the op.
template <typename T> void classify(SegOp<T> &d, size_t m) {
    const int dim = m == 1 ? 2 : 4;
    auto re = [&](const T *M, int r, int c) { return M[2 * (r * dim + c)]; };
    auto im = [&](const T *M, int r, int c) { return M[2 * (r * dim + c) + 1]; };
    bool diag = true, real = true;
    for (int r = 0; r < dim; r++) {
        for (int c = 0; c < dim; c++) {
            if (r != c && (re(d.U, r, c) != 0 || im(d.U, r, c) != 0)) {
                diag = false;
            }
            if (im(d.U, r, c) != 0) {
                real = false;
            }
        }
    }
    // A transposition of two op-local indices with unit entries.
    int moved[4], nm = 0;
    bool perm = real;
    for (int r = 0; r < dim && perm; r++) {
        int ones = 0, col = -1;
        for (int c = 0; c < dim; c++) {
            const T v = re(d.U, r, c);
            if (v == 1) {
                ones++;
                col = c;
            } else if (v != 0) {
                perm = false;
            }
        }
        perm = perm && ones == 1;
        if (perm && col != r) {
            if (nm < 4) {
                moved[nm] = r;
            }
            nm++;
        }
    }
    if (diag) {
        d.ukind = U_DIAG;
    } else if (perm && nm == 2 && re(d.U, moved[0], moved[1]) == 1) {
        d.ukind = U_SWAP;
        d.swap = 4 * moved[0] + moved[1];
    } else if (real) {
        d.ukind = U_REAL;
    } else {
        d.ukind = U_DENSE;
    }
    d.gkind = G_DENSE;
    if (d.slot >= 0) {
        bool gdiag = true;
        for (int r = 0; r < dim; r++) {
            for (int c = 0; c < dim; c++) {
                if (im(d.G, r, c) != 0 || (r != c && re(d.G, r, c) != 0)) {
                    gdiag = false;
                }
            }
        }
        bool gz = gdiag;
        for (int r = 0; r < dim && gz; r++) {
            gz = re(d.G, r, r) == ((__builtin_popcount(r) & 1) ? -1 : 1);
        }
        if (gz) {
            d.gkind = G_Z;
        } else if (gdiag) {
            d.gkind = G_DIAG;
        } else if (m == 1 && re(d.G, 0, 0) == 0 && im(d.G, 0, 0) == 0 && re(d.G, 1, 1) == 0 &&
                   im(d.G, 1, 1) == 0) {
            if (re(d.G, 0, 1) == 1 && im(d.G, 0, 1) == 0 && re(d.G, 1, 0) == 1 && im(d.G, 1, 0) == 0) {
                d.gkind = G_X;
            } else if (re(d.G, 0, 1) == 0 && im(d.G, 0, 1) == -1 && re(d.G, 1, 0) == 0 &&
                       im(d.G, 1, 0) == 1) {
                d.gkind = G_Y;
            }
        }
    }
}

template <typename T>
SegMeta build_segment(const Segment &seg, int n, std::vector<unsigned char> &table) {
    SegMeta meta;
    SegLaunch &L = meta.L;
    L.n = n;
    L.K = static_cast<int>(seg.wires.size());
    std::vector<std::pair<int, size_t>> bw; // (bit, wire)
    for (auto w : seg.wires) {
        bw.push_back({n - 1 - static_cast<int>(w), w});
    }
    std::sort(bw.begin(), bw.end());
    std::map<size_t, int> pos;
    for (int q = 0; q < L.K; q++) {
        L.bits[q] = bw[q].first;
        pos[bw[q].second] = q;
    }
    std::vector<SegOp<T>> group;
    int slot = 0;
    for (const auto &p : seg.ops) {
        SegOp<T> d{};
        d.slot = -1;
        d.m = static_cast<int32_t>(p.U.wires.size());
        const auto &w = p.U.wires;
        bool swapb = false;
        if (w.size() == 1) {
            d.cls = pos.at(w[0]);
        } else {
            int qa = pos.at(w[0]), qb = pos.at(w[1]);
            if (qa < qb) {
                std::swap(qa, qb);
                swapb = true;
            }
            if (L.K == 2) {
                d.cls = 2;
            } else {
                d.cls = (qa == 1) ? 3 : (qb == 0 ? 4 : 5);
            }
        }
        put_mat(d.U, p.U.mat, swapb);
        if (p.trainable) {
            if (p.G.wires != p.U.wires) {
                raise(PLK_ERR_INVALID, "generator wires differ from gate wires");
            }
            put_mat(d.G, p.G.mat, swapb);
            d.slot = slot;
            meta.cols[slot] = p.col;
            meta.coefs[slot] = p.coef;
            slot++;
        }
        classify(d, w.size());
        group.push_back(d);
    }
    meta.first = pack_ops(table, group.data(), group.size());
    L.nops = static_cast<int>(seg.ops.size());
    L.nslots = slot;
    return meta;
}

template <typename T>
void build_pass(const Pass &ps, int n, std::vector<unsigned char> &table,
                std::vector<TileBundle> &btab, SegMeta &meta) {
    TileLaunch &TL = meta.TL;
    TL.n = n;
    TL.T = static_cast<int>(ps.tb.size());
    for (int q = 0; q < TL.T; q++) {
        TL.tb[q] = ps.tb[q];
    }
    int pos[64];
    for (size_t q = 0; q < ps.tb.size(); q++) {
        pos[ps.tb[q]] = static_cast<int>(q);
    }
    meta.first_bundle = btab.size();
    int slot0 = 0;
    for (const auto &b : ps.bundles) {
        TileBundle tb{};
        tb.K = b.K;
        tb.qa = b.qa;
        tb.qb = b.qb;
        tb.nops = static_cast<int32_t>(b.ops.size());
        tb.nslots = b.nslots;
        tb.slot0 = slot0;
        int slot = 0;
        std::vector<SegOp<T>> group;
        for (const auto &p : b.ops) {
            SegOp<T> d{};
            d.slot = -1;
            d.m = static_cast<int32_t>(p.U.wires.size());
            const auto &w = p.U.wires;
            bool swapb = false;
            if (w.size() == 1) {
                const int q = pos[n - 1 - static_cast<int>(w[0])];
                d.cls = (b.K == 1 || q == b.qb) ? 0 : 1;
            } else {
                const int q0 = pos[n - 1 - static_cast<int>(w[0])];
                swapb = (q0 != b.qa);
                d.cls = 2;
            }
            put_mat(d.U, p.U.mat, swapb);
            if (p.trainable) {
                put_mat(d.G, p.G.mat, swapb);
                d.slot = slot++;
            }
            classify(d, w.size());
            group.push_back(d);
        }
        const size_t off = pack_ops(table, group.data(), group.size());
        if (off > static_cast<size_t>(INT32_MAX)) {
            raise(PLK_ERR_UNSUPPORTED, "operation table exceeds 2 GiB");
        }
        tb.first = static_cast<int32_t>(off);
        slot0 += b.nslots;
        btab.push_back(tb);
    }
    TL.nbundles = static_cast<int>(ps.bundles.size());
    TL.nslots = ps.nslots;
}

// Device tables of segment/pass descriptors for a whole plan (one upload).
// Host images of a plan's device tables: op groups of register segments and
// LDS bundles, the bundle table, and register-tile programs, with the
// launch metadata that points into them.
// An entry of the Jacobian formed from the sums of a register-tile pass.
struct RtTerm {
    int col;
    int slot[3]; // -1: none
    double m[3]; // coefficients, the gate's own included
};

// The instruction of an op with patched gates (batch plans).
struct RtPatch {
    size_t op;
    size_t ins;  // byte offset of its reals in the program
    int term;    // first of its terms, -1: none
    int16_t ukind, parts;
};

struct RtProgram {
    RtLaunch L{};
    std::vector<RtPatch> patches;
    size_t off = 0; // byte offset of the program in the plan blob
    std::vector<RtTerm> terms;
};

// A single-op step run by the step kernels (kernels_step.hip): its launch
// arguments, the byte offset of its U and G matrices in the image's matrix
// table, and its Jacobian column and coefficient.
struct StepMeta {
    bool ok = false;
    StepLaunch L{};
    size_t off = 0;
    int col = 0;
    double coef = 0.0;
};

// Steps first .. first + count - 1 of a plan, taken in one launch.
struct SlabGroup {
    size_t first = 0, count = 0;
    size_t off = 0; // their SlabSteps in PlanImage::mats
    SlabLaunch L{};
};

struct PlanImage {
    std::vector<SlabGroup> slabs;
    std::vector<unsigned char> ops;
    std::vector<TileBundle> bundles;
    std::vector<SegMeta> metas;
    std::vector<unsigned char> rt;
    std::vector<RtProgram> progs;
    std::vector<unsigned char> mats; // U and G of the step-kernel steps (FP64 complex)
    std::vector<StepMeta> singles;
    std::vector<RtEntry> entries; // reverse plans: see place_partials
};

// Device addresses of an image's tables.
struct PlanPlace {
    const unsigned char *ops = nullptr;
    const TileBundle *bundles = nullptr;
    const unsigned char *rt = nullptr;
    const unsigned char *mats = nullptr;
    const RtEntry *entries = nullptr;
};

// The 2^m x 2^m matrix, over the wires uw (uw[0] most significant), of an
// operator on the wires gw (a subset of uw) given as a dense matrix or as
// parity phases (even / odd); false when gw is not a subset of uw.
bool embed_matrix(const std::vector<size_t> &uw, const std::vector<size_t> &gw, OpKind kind,
                  const std::vector<cd> &gm, cd even, cd odd, std::vector<cd> &out) {
    const int m = static_cast<int>(uw.size());
    const int k = static_cast<int>(gw.size());
    const int D = 1 << m;
    std::vector<int> shift; // bit of the local index that carries gw[q]
    int gmask = 0;
    for (auto w : gw) {
        const auto it = std::find(uw.begin(), uw.end(), w);
        if (it == uw.end()) {
            return false;
        }
        shift.push_back(m - 1 - static_cast<int>(it - uw.begin()));
        gmask |= 1 << shift.back();
    }
    auto sub = [&](int r) {
        int v = 0;
        for (int q = 0; q < k; q++) {
            v |= ((r >> shift[q]) & 1) << (k - 1 - q);
        }
        return v;
    };
    out.assign(static_cast<size_t>(D) * D, cd{0.0, 0.0});
    for (int r = 0; r < D; r++) {
        for (int c = 0; c < D; c++) {
            if ((r & ~gmask) != (c & ~gmask)) {
                continue;
            }
            const int sr = sub(r), sc = sub(c);
            cd v{0.0, 0.0};
            if (kind == OpKind::Dense) {
                v = gm[static_cast<size_t>(sr) * (size_t{1} << k) + sc];
            } else if (sr == sc) {
                v = (__builtin_popcount(sr) & 1) ? odd : even;
            }
            out[static_cast<size_t>(r) * D + c] = v;
        }
    }
    return true;
}

// Fills m for a single-op step the step kernels can run: parity phases on
// any number of wires (with a parity generator when trainable) or a dense
// matrix on at most 4 wires whose generator acts inside its wires, restricted
// to the local states it moves. Appends the matrices to mats; returns false
// for anything else (the op then runs through the per-state path).
bool build_step(const PlanOp &p, int n, std::vector<unsigned char> &mats, StepMeta &m) {
    if (env_int("PLK_STEPS", 1) == 0) {
        return false;
    }
    const CompiledOp &U = p.U;
    StepLaunch L{};
    auto mask = [&](const std::vector<size_t> &w) {
        uint64_t x = 0;
        for (auto v : w) {
            x |= uint64_t{1} << (n - 1 - static_cast<int>(v));
        }
        return x;
    };
    if (U.kind == OpKind::Parity) {
        if (p.trainable && p.G.kind != OpKind::Parity) {
            return false;
        }
        L.m = 0;
        L.groups = uint64_t{1} << n;
        L.umask = mask(U.wires);
        L.gmask = p.trainable ? mask(p.G.wires) : 0;
        L.ue[0] = U.even.real();
        L.ue[1] = U.even.imag();
        L.uo[0] = U.odd.real();
        L.uo[1] = U.odd.imag();
    } else if (U.kind == OpKind::Dense && !U.wires.empty() && U.wires.size() <= STEP_MMAX) {
        const int mw = static_cast<int>(U.wires.size());
        const size_t full = size_t{1} << mw;
        std::vector<cd> gm(full * full, cd{0.0, 0.0});
        if (p.trainable &&
            !embed_matrix(U.wires, p.G.wires, p.G.kind, p.G.mat, cd{1.0, 0.0}, cd{-1.0, 0.0}, gm)) {
            return false;
        }
        // The local states the step has to touch: those where U differs
        // from the identity or G is non-zero (exact comparisons: any
        // deviation keeps a state in), padded to 2, 4, 8 or 16 with states
        // on which U is the identity and G zero.
        std::vector<size_t> act, idle;
        for (size_t k = 0; k < full; k++) {
            bool on = false;
            for (size_t c = 0; c < full && !on; c++) {
                const cd e = k == c ? cd{1.0, 0.0} : cd{0.0, 0.0};
                on = U.mat[k * full + c] != e || U.mat[c * full + k] != e ||
                     gm[k * full + c] != cd{0.0, 0.0} || gm[c * full + k] != cd{0.0, 0.0};
            }
            (on ? act : idle).push_back(k);
        }
        size_t D = 2;
        while (D < act.size()) {
            D *= 2;
        }
        for (size_t q = 0; act.size() < D; q++) {
            act.push_back(idle[q]);
        }
        L.m = mw;
        L.dim = static_cast<int>(D);
        L.groups = uint64_t{1} << (n - mw);
        std::vector<int> bits;
        for (auto w : U.wires) {
            bits.push_back(n - 1 - static_cast<int>(w));
        }
        std::vector<int> sorted = bits;
        std::sort(sorted.begin(), sorted.end());
        for (int q = 0; q < mw; q++) {
            L.bits[q] = sorted[q];
        }
        for (size_t i = 0; i < D; i++) {
            uint64_t o = 0;
            for (int q = 0; q < mw; q++) {
                if ((act[i] >> (mw - 1 - q)) & 1U) {
                    o |= uint64_t{1} << bits[q];
                }
            }
            L.off[i] = o;
        }
        mats.resize((mats.size() + 255) & ~size_t{255}, 0);
        m.off = mats.size();
        auto put = [&](const std::vector<cd> &M) {
            for (size_t r = 0; r < D; r++) {
                for (size_t c = 0; c < D; c++) {
                    const cd v = M[act[r] * full + act[c]];
                    const double re = v.real(), im = v.imag();
                    const auto *a = reinterpret_cast<const unsigned char *>(&re);
                    const auto *b = reinterpret_cast<const unsigned char *>(&im);
                    mats.insert(mats.end(), a, a + sizeof re);
                    mats.insert(mats.end(), b, b + sizeof im);
                }
            }
        };
        put(U.mat);
        put(gm);
    } else {
        return false;
    }
    L.trainable = p.trainable ? 1 : 0;
    L.write_phi = 1;
    m.L = L;
    m.col = p.col;
    m.coef = p.coef;
    m.ok = true;
    return true;
}

// Whether the step kernels run this single-op step.
bool step_kernel_ok(const PlanOp &p, int n) {
    std::vector<unsigned char> scratch;
    StepMeta m;
    return build_step(p, n, scratch, m);
}

template <typename T>
void build_seg_tables(const std::vector<Step> &steps, int n, PlanImage &img) {
    for (const auto &s : steps) {
        if (s.fused) {
            img.metas.push_back(build_segment<T>(s.seg, n, img.ops));
        } else if (s.tiled && !s.pass.rt) {
            SegMeta m;
            build_pass<T>(s.pass, n, img.ops, img.bundles, m);
            img.metas.push_back(m);
        } else {
            img.metas.push_back(SegMeta{});
        }
    }
}

// ---------------------------------------------------------------------------
// Register-tile pass programs (kernels_rtile.hip).
//
// A pass's tile bits are split into R register bits and 6 lane positions.
// An operation needs in registers the bits it mixes (bits in which its U, or
// its generator, has an entry between different values); its other bits may
// sit on lanes, where each lane applies the block its lane bits select. The
// builder picks the load layout (the first mixing bits in registers, the
// next on the lane positions from 5 down, the two cheapest to exchange
// first), then walks the ops and brings each missing mixing bit into a
// register by exchanging it with the register whose next use is farthest
// away (Belady). The final layout is the store layout.
// ---------------------------------------------------------------------------
template <typename T> struct RtBuilder {
    struct Slot {
        RtInstr h;
        T u[8];
    };
    static_assert(sizeof(Slot) == rt_stride<T>(), "instruction stride");
    std::vector<unsigned char> &blob;
    std::vector<Slot> ins;
    std::vector<unsigned char> pay;

    RtBuilder(std::vector<unsigned char> &b, size_t ops) : blob(b) { ins.reserve(ops + 2); }

    void add(const RtInstr &h, const std::vector<double> &u) {
        Slot s{};
        s.h = h;
        for (size_t k = 0; k < u.size() && k < 8; k++) {
            s.u[k] = static_cast<T>(u[k]);
        }
        ins.push_back(s);
    }

    int32_t put(const std::vector<double> &vals) {
        pay.resize((pay.size() + 15) & ~size_t{15}, 0);
        const size_t off = pay.size();
        for (double v : vals) {
            const T t = static_cast<T>(v);
            const auto *p = reinterpret_cast<const unsigned char *>(&t);
            pay.insert(pay.end(), p, p + sizeof(T));
        }
        return static_cast<int32_t>(off); // relative to the payload start; rebased in finish()
    }

    // Appends the program to the blob. One empty instruction follows the
    // last: the kernel fetches one ahead.
    size_t finish() {
        ins.push_back(Slot{});
        const size_t head = ins.size() * sizeof(Slot);
        for (auto &i : ins) {
            i.h.uoff += static_cast<int32_t>(head);
            i.h.goff += static_cast<int32_t>(head);
        }
        blob.resize((blob.size() + 255) & ~size_t{255}, 0);
        const size_t off = blob.size();
        if (off + head + pay.size() > static_cast<size_t>(INT32_MAX)) {
            raise(PLK_ERR_UNSUPPORTED, "register-tile program table exceeds 2 GiB");
        }
        const auto *pi = reinterpret_cast<const unsigned char *>(ins.data());
        blob.insert(blob.end(), pi, pi + head);
        blob.insert(blob.end(), pay.begin(), pay.end());
        return off;
    }
};

std::vector<double> cplx(const std::vector<cd> &v) {
    std::vector<double> out;
    out.reserve(2 * v.size());
    for (auto &x : v) {
        out.push_back(x.real());
        out.push_back(x.imag());
    }
    return out;
}

bool is_real(const std::vector<cd> &v) {
    for (auto &x : v) {
        if (x.imag() != 0.0) {
            return false;
        }
    }
    return true;
}

// 2x2 block of a 4x4 op matrix over local bit `lr` (the register wire) with
// the other local bit fixed to c.
std::vector<cd> block2(const std::vector<cd> &M, int lr, int c) {
    std::vector<cd> B(4);
    for (int x = 0; x < 2; x++) {
        for (int y = 0; y < 2; y++) {
            const int r = lr == 1 ? (2 * x + c) : (2 * c + x);
            const int col = lr == 1 ? (2 * y + c) : (2 * c + y);
            B[2 * x + y] = M[4 * r + col];
        }
    }
    return B;
}

bool is_diag2(const std::vector<cd> &B) { return B[1] == cd(0, 0) && B[2] == cd(0, 0); }
bool is_ident2(const std::vector<cd> &B) {
    return B[0] == cd(1, 0) && B[3] == cd(1, 0) && is_diag2(B);
}
bool is_x2(const std::vector<cd> &B) {
    return B[0] == cd(0, 0) && B[3] == cd(0, 0) && B[1] == cd(1, 0) && B[2] == cd(1, 0);
}

// Encodes the U part of a one-register-bit op; returns its reals. ukind: the
// kind of a batch run (its reals are patched), -1: the matrix's.
std::vector<double> rt_encode_u1(RtInstr &in, const std::vector<cd> &U, int ukind) {
    if (ukind < 0) {
        ukind = is_ident2(U) ? U_NONE : is_diag2(U) ? U_DIAG : is_x2(U) ? U_SWAP : is_real(U) ? U_REAL : U_DENSE;
    }
    in.ukind = static_cast<int8_t>(ukind);
    switch (ukind) {
    case U_DIAG:
        return cplx({U[0], U[3]});
    case U_REAL:
        return {U[0].real(), U[1].real(), U[2].real(), U[3].real()};
    case U_DENSE:
        return cplx(U);
    default:
        return {};
    }
}

// complex64 programs round every matrix to FP32, which changes the norm of
// the whole state by a few 1e-8 per gate: the one rounding error that does not
// average out over the amplitudes (its random walk over a circuit's gates is
// the bulk of an FP32 expectation value's error). `norm` is the product of
// these factors so far, the norms of the rounded matrices by those of the given
// ones (which need not be unitary); a one-wire matrix is divided by it before it
// is rounded, so the product stays within one rounding of 1. A matrix of zeros or
// of numbers that FP32 does not hold is left as it is.
std::vector<double> keep_norm(const std::vector<double> &u, double &norm) {
    std::vector<double> v = u;
    double given = 0.0, rounded = 0.0;
    for (size_t k = 0; k < u.size(); k++) {
        v[k] = u[k] / norm;
        const double r = static_cast<double>(static_cast<float>(v[k]));
        given += u[k] * u[k];
        rounded += r * r;
    }
    const double next = norm * std::sqrt(rounded / given);
    if (!(std::abs(next - 1.0) < 1e-6)) {
        return u;
    }
    norm = next;
    return v;
}

// Index bits that sit on lanes at load and store (complex128: bit 0, complex64:
// bits 0 and 1), so that every load and store instruction covers runs of at
// least 32 bytes. With the three lowest bits all in registers each instruction
// touches 64 cache lines 16 bytes at a time, and an in-place pass streams at 4.4
// TB/s instead of 5.1 (1-4 GiB states). A keep bit the pass mixes is swapped into
// a register when an op needs it.
int keep_bits(int dtype) { return dtype == PLK_C64 ? 2 : 1; }

// The state bits of an op of at most two wires.
struct BitList {
    int bit[2];
    int count = 0;
    void push_back(int b) { bit[count++] = b; }
    const int *begin() const { return bit; }
    const int *end() const { return bit + count; }
    int size() const { return count; }
    int operator[](int k) const { return bit[k]; }
};

template <typename T>
RtProgram build_rt_program(const Pass &ps, int n, int R, int keep, std::vector<unsigned char> &blob, double &norm,
                           bool patched = false) {
    RtProgram out;
    RtLaunch &L = out.L;
    L.n = n;
    L.R = R;
    L.wide = sizeof(T) == 8 ? 1 : 0;
    L.T = static_cast<int>(ps.tb.size());
    if (L.T != R + RT_LANE_BITS) {
        raise(PLK_ERR_INVALID, "register-tile pass of the wrong width");
    }
    for (int q = 0; q < L.T; q++) {
        L.tb[q] = ps.tb[q];
    }
    const size_t nops = ps.ops.size();
    std::vector<BitList> gbits(nops), mix(nops);
    std::vector<Place> place(nops);
    for (size_t i = 0; i < nops; i++) {
        const PlanOp &p = ps.ops[i];
        const uint64_t mm = place[i].mix = p.mix;
        place[i].trainable = p.trainable;
        place[i].skew = p.skew;
        for (auto w : p.U.wires) {
            const int gb = n - 1 - static_cast<int>(w);
            gbits[i].push_back(gb);
            place[i].on |= uint64_t{1} << gb;
            if (mm >> gb & 1) {
                mix[i].push_back(gb);
            }
        }
    }
    // Load layout.
    std::vector<int> order;
    for (size_t i = 0; i < nops; i++) {
        for (int q : mix[i]) {
            if (std::find(order.begin(), order.end(), q) == order.end()) {
                order.push_back(q);
            }
        }
    }
    // The lowest `keep` index bits sit on lanes at load and store.
    auto is_keep = [&](int q) { return q < keep; };
    auto has = [](const std::vector<int> &v, int q) { return std::find(v.begin(), v.end(), q) != v.end(); };
    std::vector<int> reg, lane(RT_LANE_BITS, -1), hot;
    for (int q : order) {
        if (!is_keep(q) && static_cast<int>(reg.size()) < R) {
            reg.push_back(q);
        } else {
            hot.push_back(q);
        }
    }
    std::vector<int> rest;
    for (int q : ps.tb) {
        if (!has(reg, q) && !has(hot, q)) {
            rest.push_back(q); // ascending global bits
        }
    }
    while (static_cast<int>(reg.size()) < R) {
        // Fill registers with the highest remaining bits, never a keep bit.
        reg.push_back(rest.back());
        rest.pop_back();
    }
    for (size_t k = 0; k < hot.size(); k++) {
        lane[5 - k] = hot[k];
    }
    for (int p = 0, r = 0; p < RT_LANE_BITS; p++) {
        if (lane[p] < 0) {
            lane[p] = rest[r++];
        }
    }
    for (int r = 0; r < R; r++) {
        L.reg_in[r] = reg[r];
    }
    for (int p = 0; p < RT_LANE_BITS; p++) {
        L.lane_in[p] = lane[p];
    }

    RtBuilder<T> b(blob, nops);
    auto reg_of = [&](int q) {
        for (int r = 0; r < R; r++) {
            if (reg[r] == q) {
                return r;
            }
        }
        return -1;
    };
    auto lane_of = [&](int q) {
        for (int p = 0; p < RT_LANE_BITS; p++) {
            if (lane[p] == q) {
                return p;
            }
        }
        raise(PLK_ERR_INVALID, "register-tile op outside the tile bits");
    };
    // Selector of a non-mixing bit: its lane position, or 64 + the bit when
    // it lies outside the tile (fixed for the whole tile).
    auto sel_of = [&](int q) -> int {
        for (int p = 0; p < RT_LANE_BITS; p++) {
            if (lane[p] == q) {
                return p;
            }
        }
        if (std::find(ps.tb.begin(), ps.tb.end(), q) != ps.tb.end()) {
            raise(PLK_ERR_INVALID, "register-tile selector bit sits in a register");
        }
        return 64 + q;
    };
    auto add_remap = [&](RtInstr &in, int r, int p) {
        if (in.nremap >= 2) {
            raise(PLK_ERR_INVALID, "register-tile instruction needs more than two remaps");
        }
        if (in.nremap == 0) {
            in.rq0 = static_cast<int8_t>(r);
            in.rp0 = static_cast<int8_t>(p);
        } else {
            in.rq1 = static_cast<int8_t>(r);
            in.rp1 = static_cast<int8_t>(p);
        }
        in.nremap++;
        std::swap(lane[p], reg[r]);
    };
    int slot = 0;
    // Operations leave in an order that commutes with the pass's: first all
    // whose mixed bits sit in registers, then the first left, with its bits
    // exchanged for the register bits that are needed last. In the pass's own
    // order half as many again are needed (24-qubit Jacobian: 180 in 29 passes,
    // now 117; 12 qubits 52, now 31), each 64 to 192 vector instructions of a
    // four-state program: 12-qubit Jacobian of 12 observables 389 to 373 us,
    // larger ones, which wait for memory, the same.
    std::vector<size_t> left(nops);
    for (size_t i = 0; i < nops; i++) {
        left[i] = i;
    }
    size_t scan = 0; // left[0 .. scan) wait for registers or for each other
    Blocked blocked;
    while (!left.empty()) {
        size_t at = 0;
        for (; scan < left.size(); scan++) {
            const size_t k = left[scan];
            if (!blocked.stops(place[k]) &&
                std::all_of(mix[k].begin(), mix[k].end(), [&](int q) { return reg_of(q) >= 0; })) {
                at = scan;
                break;
            }
            blocked.add(place[k]);
        }
        const bool stuck = scan == left.size();
        const size_t i = left[at];
        left.erase(left.begin() + static_cast<long>(at));
        if (stuck) {
            scan = 0;
            blocked = Blocked{};
        }
        const PlanOp &p = ps.ops[i];
        RtInstr in{};
        in.slot = -1;
        in.s0 = in.s1 = -1;
        std::vector<double> u;
        for (int q : mix[i]) {
            if (reg_of(q) >= 0) {
                continue;
            }
            int victim = -1;
            size_t far = 0;
            for (int r = 0; r < R; r++) {
                if (std::find(mix[i].begin(), mix[i].end(), reg[r]) != mix[i].end()) {
                    continue;
                }
                size_t use = 0;
                while (use < left.size() && !(place[left[use]].mix >> reg[r] & 1)) {
                    use++;
                }
                if (victim < 0 || use > far) {
                    victim = r;
                    far = use;
                }
            }
            add_remap(in, victim, lane_of(q));
        }
        const int m = gbits[i].size();
        const std::vector<cd> *G = nullptr;
        const int term0 = static_cast<int>(out.terms.size());
        if (p.trainable) {
            in.slot = slot;
            if (p.run.empty()) {
                if (p.G.wires != p.U.wires || p.G.kind != OpKind::Dense) {
                    raise(PLK_ERR_INVALID, "generator wires differ from gate wires");
                }
                G = &p.G.mat;
                out.terms.push_back({p.col, {slot, -1, -1}, {p.coef, 0.0, 0.0}});
            } else {
                const int parts = run_parts(p);
                const bool all = rt_slots(p) == 3;
                const int only = parts == 1 ? 0 : parts == 2 ? 1 : 2;
                in.gkind = static_cast<int8_t>(all ? G_XYZ : only == 0 ? G_X : only == 1 ? G_Y : G_Z);
                for (const RunTerm &t : p.run) {
                    if (all) {
                        out.terms.push_back({t.col, {slot, slot + 1, slot + 2},
                                             {t.coef * t.m[0], t.coef * t.m[1], t.coef * t.m[2]}});
                    } else {
                        out.terms.push_back({t.col, {slot, -1, -1}, {t.coef * t.m[only], 0.0, 0.0}});
                    }
                }
            }
            slot += rt_slots(p);
        }
        if (m == 1) {
            const int r = reg_of(gbits[i][0]);
            if (r >= 0) {
                in.code = RT_REG1;
                in.a = static_cast<int8_t>(r);
                u = rt_encode_u1(in, p.U.mat, p.ukind);
                if (sizeof(T) == 4 && !u.empty() && !patched) {
                    u = keep_norm(u, norm);
                }
                if (G) {
                    const auto &g = *G;
                    if (is_diag2(g) && is_real(g)) {
                        in.gkind = G_DIAG;
                        in.goff = b.put({g[0].real(), g[3].real()});
                    } else {
                        in.gkind = G_DENSE;
                        in.goff = b.put(cplx(g));
                    }
                }
            } else {
                in.code = RT_LANE;
                in.s0 = static_cast<int8_t>(sel_of(gbits[i][0]));
                u = cplx({p.U.mat[0], p.U.mat[3]});
                if (sizeof(T) == 4 && !patched) {
                    u = keep_norm(u, norm);
                }
                if (G) {
                    in.goff = b.put({(*G)[0].real(), (*G)[3].real()});
                } else if (p.trainable) {
                    in.goff = b.put({1.0, -1.0}); // a diagonal run: Z
                }
            }
        } else {
            const int r0 = reg_of(gbits[i][0]), r1 = reg_of(gbits[i][1]);
            if (r0 >= 0 && r1 >= 0) {
                in.code = RT_REG2;
                in.a = static_cast<int8_t>(std::max(r0, r1));
                in.b = static_cast<int8_t>(std::min(r0, r1));
                SegOp<double> d{};
                d.slot = G ? 0 : -1;
                put_mat(d.U, p.U.mat, r0 < r1);
                if (G) {
                    put_mat(d.G, *G, r0 < r1);
                }
                classify(d, 2);
                in.ukind = static_cast<int8_t>(d.ukind);
                in.swap = static_cast<int8_t>(d.swap);
                if (d.ukind == U_DIAG) {
                    for (int k = 0; k < 4; k++) {
                        u.push_back(d.U[2 * (5 * k)]);
                        u.push_back(d.U[2 * (5 * k) + 1]);
                    }
                } else if (d.ukind == U_REAL) {
                    std::vector<double> v;
                    for (int e = 0; e < 16; e++) {
                        v.push_back(d.U[2 * e]);
                    }
                    in.uoff = b.put(v);
                } else if (d.ukind == U_DENSE) {
                    in.uoff = b.put(std::vector<double>(d.U, d.U + 32));
                }
                if (G) {
                    in.gkind = static_cast<int8_t>(d.gkind);
                    std::vector<double> g;
                    if (d.gkind == G_DIAG) {
                        for (int k = 0; k < 4; k++) {
                            g.push_back(d.G[2 * (5 * k)]);
                        }
                    } else if (d.gkind == G_DENSE) {
                        g.assign(d.G, d.G + 32);
                    }
                    in.goff = b.put(g);
                }
            } else if (r0 >= 0 || r1 >= 0) {
                // One wire on a register bit, the other (not mixed) on a lane.
                const int k_reg = r0 >= 0 ? 0 : 1;
                const int lr = 1 - k_reg; // local bit of the register wire
                in.code = RT_SEL;
                in.a = static_cast<int8_t>(k_reg == 0 ? r0 : r1);
                in.s0 = static_cast<int8_t>(sel_of(gbits[i][1 - k_reg]));
                const std::vector<cd> B0 = block2(p.U.mat, lr, 0), B1 = block2(p.U.mat, lr, 1);
                if (is_diag2(B0) && is_diag2(B1)) {
                    in.ukind = U_DIAG;
                    u = cplx({B0[0], B0[3], B1[0], B1[3]});
                } else if ((is_ident2(B0) || is_x2(B0)) && (is_ident2(B1) || is_x2(B1))) {
                    in.ukind = U_SWAP;
                    u = {is_x2(B0) ? 1.0 : 0.0, is_x2(B1) ? 1.0 : 0.0};
                } else if (is_real(B0) && is_real(B1)) {
                    in.ukind = U_REAL;
                    u = {B0[0].real(), B0[1].real(), B0[2].real(), B0[3].real(),
                         B1[0].real(), B1[1].real(), B1[2].real(), B1[3].real()};
                } else {
                    in.ukind = U_DENSE;
                    std::vector<double> v = cplx(B0), v1 = cplx(B1);
                    v.insert(v.end(), v1.begin(), v1.end());
                    in.uoff = b.put(v);
                }
                if (G) {
                    const std::vector<cd> G0 = block2(*G, lr, 0), G1 = block2(*G, lr, 1);
                    if (is_diag2(G0) && is_diag2(G1) && is_real(G0) && is_real(G1)) {
                        in.gkind = G_DIAG;
                        in.goff = b.put({G0[0].real(), G0[3].real(), G1[0].real(), G1[3].real()});
                    } else {
                        in.gkind = G_DENSE;
                        std::vector<double> g = cplx(G0), g1 = cplx(G1);
                        g.insert(g.end(), g1.begin(), g1.end());
                        in.goff = b.put(g);
                    }
                }
            } else {
                // Both wires on lanes: diagonal; block c = bit(wires[1]) + 2 bit(wires[0]) is
                // the op's local index.
                in.code = RT_LANE;
                in.s0 = static_cast<int8_t>(sel_of(gbits[i][1]));
                in.s1 = static_cast<int8_t>(sel_of(gbits[i][0]));
                std::vector<cd> f;
                for (int k = 0; k < 4; k++) {
                    f.push_back(p.U.mat[5 * k]);
                }
                u = cplx(f);
                if (G) {
                    std::vector<double> g;
                    for (int k = 0; k < 4; k++) {
                        g.push_back((*G)[5 * k].real());
                    }
                    in.goff = b.put(g);
                }
            }
        }
        if (patched) {
            bool any = false;
            for (const RunGate &g : p.gates) {
                any = any || g.g.gate != BPG_CONST;
            }
            if (any) {
                const int parts = run_parts(p);
                out.patches.push_back({i, b.ins.size() * rt_stride<T>() + sizeof(RtInstr),
                                       p.run.empty() ? -1 : term0,
                                       static_cast<int16_t>(in.code == RT_LANE ? U_DIAG : in.ukind),
                                       static_cast<int16_t>(rt_slots(p) == 3 ? 7 : parts)});
            }
        }
        b.add(in, u);
    }
    // Store layout: keep bits left in registers go back to lanes, to the
    // highest position (the cheapest exchange) that holds no keep bit.
    RtInstr fin{};
    fin.slot = -1;
    for (int q = 0; q < keep; q++) {
        const int r = reg_of(q);
        if (r < 0) {
            continue;
        }
        int p = RT_LANE_BITS - 1;
        while (is_keep(lane[p])) {
            p--;
        }
        add_remap(fin, r, p);
    }
    if (fin.nremap > 0) {
        b.add(fin, {});
    }
    for (int r = 0; r < R; r++) {
        L.reg_out[r] = reg[r];
    }
    for (int p = 0; p < RT_LANE_BITS; p++) {
        L.lane_out[p] = lane[p];
    }
    L.ninstr = static_cast<int>(b.ins.size());
    L.nslots = slot;
    if (slot > RT_SLOTS_MAX) {
        raise(PLK_ERR_INVALID, "register-tile pass with too many sums");
    }
    out.off = b.finish();
    return out;
}

// Whether a two-wire op leaves two of its four local states alone, in its
// matrix and in its generator: as a single-op step it moves half a state.
bool moves_half(const PlanOp &p) {
    if (p.U.wires.size() != 2 || !p.run.empty() || (p.trainable && p.G.wires != p.U.wires)) {
        return false;
    }
    int on = 0;
    for (size_t k = 0; k < 4; k++) {
        bool act = false;
        for (size_t c = 0; c < 4 && !act; c++) {
            const cd e = k == c ? cd{1.0, 0.0} : cd{0.0, 0.0};
            act = p.U.mat[k * 4 + c] != e || p.U.mat[c * 4 + k] != e ||
                  (p.trainable && (p.G.mat[k * 4 + c] != cd{0.0, 0.0} || p.G.mat[c * 4 + k] != cd{0.0, 0.0}));
        }
        on += act ? 1 : 0;
    }
    return on <= 2;
}

// Register-tile passes of one or two ops that move half a state each: as
// single-op steps they move no more bytes (a pass reads and writes every
// amplitude, a step only those its op moves). Between the 3-4-wire gates of a
// chemistry circuit a pass often holds one SingleExcitation: 20 qubits
// complex128, five observables, 35.6 us as a pass, 17.4 as a step.
//
// beside: only passes next to a single-op step, with which they share a launch. A
// forward pass moves one state, and alone (the last pass of a gate stream) it is
// no slower than its steps while launches count: complex64, 18 qubits, 20 gates 48
// us as a pass, 51 as steps; complex64, 13 qubits, 60 gates 89 and 103; complex128,
// 13 qubits, 600 gates 669 and 714.
void split_sparse_passes(std::vector<Step> &steps, int n, bool beside) {
    if (env_int("PLK_STEPS", 1) == 0) {
        return;
    }
    std::vector<Step> out;
    out.reserve(steps.size());
    std::vector<char> single(steps.size() + 2, 0);
    for (size_t i = 0; i < steps.size(); i++) {
        single[i + 1] = steps[i].tiled || steps[i].fused ? 0 : 1;
    }
    for (size_t i = 0; i < steps.size(); i++) {
        Step &st = steps[i];
        bool ok = st.tiled && st.pass.rt && st.pass.ops.size() <= 2 && (!beside || single[i] || single[i + 2]);
        for (size_t k = 0; ok && k < st.pass.ops.size(); k++) {
            ok = moves_half(st.pass.ops[k]) && step_kernel_ok(st.pass.ops[k], n);
        }
        if (!ok) {
            out.push_back(std::move(st));
            continue;
        }
        for (PlanOp &p : st.pass.ops) {
            Step s;
            s.single = std::move(p);
            out.push_back(std::move(s));
        }
    }
    steps.swap(out);
}

// Programs of every register-tile pass of a plan, uploaded as one blob.
// R: register bits of the tile passes.
// Groups consecutive two-state steps whose wires fit kSlabBits bits together
// with the lowest ones (whole cache lines).
void build_slabs(PlanImage &img, int n, int dtype) {
    const int S = std::min(n, kSlabBits);
    const uint64_t low = (uint64_t{1} << std::min(n, low_bits(dtype))) - 1;
    // The partials of a launch lie side by side: at most 2^26 doubles for SEG_NJMAX observables.
    const size_t most = std::min<size_t>(64, std::max<size_t>(2, (size_t{1} << 26) >> std::min(63, n - S + 3)));
    auto takes = [&](size_t i) { return img.singles[i].ok && img.singles[i].L.m > 0 && img.singles[i].L.dim == 2; };
    for (size_t i = 0; i < img.singles.size();) {
        uint64_t bits = low;
        size_t end = i;
        for (; end < img.singles.size() && end - i < most && takes(end); end++) {
            uint64_t with = bits;
            for (int q = 0; q < img.singles[end].L.m; q++) {
                with |= uint64_t{1} << img.singles[end].L.bits[q];
            }
            if (__builtin_popcountll(with) > S) {
                break;
            }
            bits = with;
        }
        if (end - i < 2) {
            i = std::max(end, i + 1);
            continue;
        }
        for (int b = 0; __builtin_popcountll(bits) < S; b++) {
            bits |= uint64_t{1} << b;
        }
        SlabGroup g;
        g.first = i;
        g.count = end - i;
        g.L.n = n;
        g.L.S = S;
        g.L.nsteps = static_cast<int>(g.count);
        for (int b = 0, q = 0; b < n; b++) {
            if (bits >> b & 1) {
                g.L.sb[q++] = b;
            }
        }
        img.mats.resize((img.mats.size() + 255) & ~size_t{255}, 0);
        g.off = img.mats.size();
        for (; i < end; i++) {
            const StepMeta &m = img.singles[i];
            SlabStep p{};
            p.off0 = m.L.off[0];
            p.off1 = m.L.off[1];
            p.mats = m.off;
            p.m = m.L.m;
            for (int q = 0; q < m.L.m; q++) {
                p.lb[q] = static_cast<int32_t>(std::find(g.L.sb, g.L.sb + S, m.L.bits[q]) - g.L.sb);
            }
            p.trainable = m.L.trainable;
            const auto *b = reinterpret_cast<const unsigned char *>(&p);
            img.mats.insert(img.mats.end(), b, b + sizeof p);
        }
        img.slabs.push_back(g);
    }
}

const SlabGroup *slab_of(const PlanImage &img, size_t i) {
    auto g = std::upper_bound(img.slabs.begin(), img.slabs.end(), i,
                              [](size_t at, const SlabGroup &x) { return at < x.first; });
    if (g == img.slabs.begin() || i >= std::prev(g)->first + std::prev(g)->count) {
        return nullptr;
    }
    return &*std::prev(g);
}

// wide: register-tile programs in FP64 for complex64 states too, which are then
// rounded once a pass instead of at every operation (forward passes only). A
// pass-by-pass program whose result is the state takes it: an expectation value of
// a 22-qubit, 4-layer circuit is a third as far from 64 bits as with a rounding per
// operation (3.4e-7 against 8.6e-7 relative). 400 gates complex64: 22 qubits 0.82
// -> 0.92 ms, 26 qubits 5.5 -> 7.2 ms. The forward run of a Jacobian, whose reverse
// sweep rounds anyway, stays in FP32, and so do states that run whole in one launch
// (at most 12 qubits), which round at every operation.
PlanImage build_image(const std::vector<Step> &steps, const State &s, bool wide) {
    PlanImage img;
    if (s.dtype == PLK_C64) {
        build_seg_tables<float>(steps, s.n, img);
    } else {
        build_seg_tables<double>(steps, s.n, img);
    }
    img.singles.resize(steps.size());
    for (size_t i = 0; i < steps.size(); i++) {
        if (!steps[i].fused && !steps[i].tiled) {
            build_step(steps[i].single, s.n, img.mats, img.singles[i]);
        }
    }
    build_slabs(img, s.n, s.dtype);
    img.progs.resize(steps.size());
    double norm = 1.0;
    for (size_t i = 0; i < steps.size(); i++) {
        if (steps[i].tiled && steps[i].pass.rt) {
            const int R = static_cast<int>(steps[i].pass.tb.size()) - RT_LANE_BITS;
            const int keep = keep_bits(s.dtype);
            img.progs[i] = s.dtype == PLK_C64 && !wide
                               ? build_rt_program<float>(steps[i].pass, s.n, R, keep, img.rt, norm)
                               : build_rt_program<double>(steps[i].pass, s.n, R, keep, img.rt, norm);
        }
    }
    return img;
}

size_t image_bytes(const PlanImage &img) {
    auto up = [](size_t x) { return (x + 255) & ~size_t{255}; };
    return up(img.ops.size()) + up(img.bundles.size() * sizeof(TileBundle)) + up(img.rt.size()) +
           up(img.mats.size()) + up(img.entries.size() * sizeof(RtEntry));
}

// Copies the image's tables to base (image_bytes(img) bytes) on the device's
// stream; the image must stay alive until the stream has run the copies.
PlanPlace copy_image(Device &dev, const PlanImage &img, unsigned char *base) {
    auto up = [](size_t x) { return (x + 255) & ~size_t{255}; };
    PlanPlace pl;
    size_t off = 0;
    auto put = [&](const void *src, size_t bytes) -> unsigned char * {
        unsigned char *dst = base + off;
        if (bytes) {
            PLK_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, dev.stream));
        }
        off += up(bytes);
        return dst;
    };
    pl.ops = put(img.ops.data(), img.ops.size());
    pl.bundles = reinterpret_cast<const TileBundle *>(
        put(img.bundles.data(), img.bundles.size() * sizeof(TileBundle)));
    pl.rt = put(img.rt.data(), img.rt.size());
    pl.mats = put(img.mats.data(), img.mats.size());
    pl.entries = reinterpret_cast<const RtEntry *>(put(img.entries.data(), img.entries.size() * sizeof(RtEntry)));
    return pl;
}

// The addresses copy_image(dev, img, base) fills, without copying.
PlanPlace place_addresses(const PlanImage &img, unsigned char *base) {
    auto up = [](size_t x) { return (x + 255) & ~size_t{255}; };
    PlanPlace pl;
    pl.ops = base;
    pl.bundles = reinterpret_cast<const TileBundle *>(base + up(img.ops.size()));
    pl.rt = base + up(img.ops.size()) + up(img.bundles.size() * sizeof(TileBundle));
    pl.mats = pl.rt + up(img.rt.size());
    pl.entries = reinterpret_cast<const RtEntry *>(pl.mats + up(img.mats.size()));
    return pl;
}

PlanPlace place_in_arena(Device &dev, const PlanImage &img) {
    const size_t bytes = image_bytes(img);
    return copy_image(dev, img, static_cast<unsigned char *>(arena_alloc(dev, bytes ? bytes : 256)));
}

// Everything a replay of the plan's launches takes as kernel arguments:
// equal signatures mean equal launches, whatever the matrices in the tables.
void append_signature(const PlanImage &img, std::vector<unsigned char> &sig) {
    auto put = [&](const void *p, size_t bytes) {
        const auto *b = static_cast<const unsigned char *>(p);
        sig.insert(sig.end(), b, b + bytes);
    };
    const uint64_t sizes[5] = {img.ops.size(), img.bundles.size(), img.rt.size(), img.mats.size(),
                               img.entries.size()};
    put(sizes, sizeof sizes);
    for (const SlabGroup &g : img.slabs) {
        put(&g.first, sizeof g.first);
        put(&g.count, sizeof g.count);
        put(&g.off, sizeof g.off);
        put(&g.L, sizeof g.L);
    }
    for (const StepMeta &m : img.singles) {
        put(&m.ok, sizeof m.ok);
        put(&m.L, sizeof m.L);
        put(&m.off, sizeof m.off);
        put(&m.col, sizeof m.col);
        put(&m.coef, sizeof m.coef);
    }
    for (const SegMeta &m : img.metas) {
        put(&m.L, sizeof m.L);
        put(&m.first, sizeof m.first);
        put(m.cols, sizeof m.cols);
        put(m.coefs, sizeof m.coefs);
        put(&m.TL, sizeof m.TL);
        put(&m.first_bundle, sizeof m.first_bundle);
    }
    for (const RtProgram &p : img.progs) {
        put(&p.L, sizeof p.L);
        put(&p.off, sizeof p.off);
    }
}

// Observable states per register-tile chunk: 3 keeps phi plus three states
// in the registers of three wavefronts per SIMD. When a pass has fewer
// tiles than the device has CUs, chunks of one state give the launch more
// blocks (12 qubits complex128, 12 observables: 0.63 ms per Jacobian against
// 0.74 with chunks of 3). PLK_RTILE_NJ overrides, up to RT_NJMAX.
int rtile_chunk(int dtype, int n, int num_cus) {
    const int e = env_int("PLK_RTILE_NJ", 0);
    if (e > 0) {
        return std::min(RT_NJMAX, e);
    }
    const int T = rt_reg_max(dtype, 3) + RT_LANE_BITS;
    const bool few_tiles = n - T < 30 && (int64_t{1} << std::max(0, n - T)) < num_cus;
    return few_tiles ? 1 : 3;
}

// Observable states of the widest chunk of a sweep.
int sweep_chunk(int dtype, int n, size_t n_obs, int num_cus) {
    return chunk_sizes(n_obs, rtile_chunk(dtype, n, num_cus)).front();
}

// Register-tile passes serve every state of at least one register tile:
// with their observable chunks side by side they measured faster than the
// LDS tile passes at every size from 10 to 21 qubits in both precisions
// (6-layer adjoint, 9 observables, complex128: 0.70 vs 2.52 ms at 10 qubits,
// 1.32 vs 2.12 at 16, 8.35 vs 11.26 at 21). PLK_RTILE=0 turns them off.
bool use_rtile(int n, int dtype, int nj) {
    return env_int("PLK_RTILE", -1) != 0 && n >= rt_reg_min(dtype, nj) + RT_LANE_BITS;
}

// Register bits of a plan's tiles. Wider tiles take fewer passes, narrower ones
// spread a pass over more wavefronts that each walk less: a pass of a few tiles
// takes as long as one wavefront needs for its program. Measured, forward
// (400-gate stream, R = 3 / 4 / 5): 15 qubits complex128 553 / 590 / 661 us, 20
// qubits 757 / 763 / 838, 22 qubits 1139 / 976 / 1023, 24 qubits 3133 / 2701 /
// 2635; 20 qubits complex64 630 / 612 / 680, 24 qubits 2407 / 1914 / 1728. One
// observable a chunk (R = 3 / 4): 17 qubits complex64, 5 observables 742 / 766 us
// (R = 5: 897); 16 qubits complex128, 9 observables 636 / 675; one observable,
// 20 qubits complex128 3208 / 3320, 21 qubits 3828 / 3673. The complex64 figures are
// those of FP32 programs. A wide one (see build_image) is bound by its FP64
// exchanges before memory, and R = 5 has fewest of them: it pays from eight tiles
// a CU on (streams of 200 gates, R = 4 / 5: 21 qubits 374 / 427 us, 22 qubits 454 /
// 448, 23 qubits 690 / 629, 24 qubits 1168 / 1062).
int plan_reg_bits(int n, int dtype, int nj, size_t chunks, int num_cus, bool wide) {
    const int lo = rt_reg_min(dtype, nj);
    int R = std::min(rt_reg_max(dtype, nj), n - RT_LANE_BITS);
    auto tiles_per_cu = [&] { return std::ldexp(static_cast<double>(chunks), n - R - RT_LANE_BITS) / num_cus; };
    const double widest = wide && dtype == PLK_C64 ? 8.0 : 32.0;
    while (R > lo && tiles_per_cu() < (R == 5 ? widest : nj == 1 ? 8.0 : 2.0)) {
        R--;
    }
    return R;
}

void apply_single(Device &dev, const State &s, const CompiledOp &op);

// Launches a forward plan whose tables are at pl (no host synchronisation
// unless a step is a single op outside the fused kernels).
void enqueue_forward(Device &dev, const State &s, const std::vector<Step> &steps,
                     const PlanImage &img, const PlanPlace &pl) {
    size_t next_slab = 0;
    for (size_t i = 0; i < steps.size(); i++) {
        if (next_slab < img.slabs.size() && img.slabs[next_slab].first == i) {
            const SlabGroup &g = img.slabs[next_slab++];
            launch_slab_steps(dev, s, nullptr, pl.mats, pl.mats + g.off, g.L, nullptr);
            i += g.count - 1;
            continue;
        }
        if (steps[i].tiled && steps[i].pass.rt) {
            RtLaunch L = img.progs[i].L;
            L.nj = 0;
            L.nc = L.nbig = 1;
            L.write_phi = 1;
            L.nslots = 0;
            launch_rtile(dev, s, nullptr, nullptr, pl.rt + img.progs[i].off, L, nullptr);
        } else if (steps[i].fused) {
            SegLaunch L = img.metas[i].L;
            L.write_phi = 1;
            L.nj = 0;
            L.nslots = 0;
            launch_segment(dev, s, nullptr, pl.ops + img.metas[i].first, L);
        } else if (steps[i].tiled) {
            TileLaunch TL = img.metas[i].TL;
            TL.nj = 0;
            TL.write_phi = 1;
            TL.nslots = 0;
            launch_tile(dev, s, nullptr, pl.bundles + img.metas[i].first_bundle, pl.ops, TL);
        } else if (img.singles[i].ok) {
            StepLaunch L = img.singles[i].L;
            L.nj = 0;
            L.trainable = 0;
            L.write_phi = 1;
            launch_step(dev, s, nullptr, pl.mats + img.singles[i].off, L, nullptr);
        } else {
            apply_single(dev, s, steps[i].single.U);
        }
    }
}

void run_forward(Device &dev, const State &s, const std::vector<Step> &steps) {
    const PlanImage img = build_image(steps, s, true);
    enqueue_forward(dev, s, steps, img, place_in_arena(dev, img));
    // The host image is read by the stream's copies.
    PLK_HIP(hipStreamSynchronize(dev.stream));
}

void apply_single(Device &dev, const State &s, const CompiledOp &op) {
    switch (op.kind) {
    case OpKind::Identity:
        return;
    case OpKind::Parity:
        launch_parity(dev, s, op.wires, op.even, op.odd);
        return;
    case OpKind::Dense:
        if (op.wires.size() <= 2) {
            PlanOp p;
            p.U = op;
            std::vector<PlanOp> v;
            v.push_back(std::move(p));
            run_forward(dev, s, plan_steps(std::move(v)));
        } else {
            launch_dense(dev, s, op);
        }
        return;
    }
}

void apply_generator_dev(Device &dev, const State &s, const CompiledGen &g) {
    if (g.kind == OpKind::Parity) {
        launch_parity(dev, s, g.wires, 1.0, -1.0);
    } else {
        launch_dense_matrix(dev, s, g.wires, g.mat);
    }
}

// ---------------------------------------------------------------------------
// Observable application and expectation values.
// ---------------------------------------------------------------------------
void apply_obs_general(Device &dev, const State &s, const ObsNode &o);

const PauliDevice *ObsNode::pauli_on(Device &dev, int n) const {
    auto it = pauli_dev.find({dev.id, n});
    if (it != pauli_dev.end()) {
        return it->second.get();
    }
    std::vector<PauliTerm> terms;
    if (!to_pauli(*this, n, terms)) {
        return nullptr;
    }
    auto &slot = pauli_dev[{dev.id, n}];
    slot = pauli_device(dev, terms);
    return slot.get();
}

void check_sparse_wires(const ObsNode &o, const State &s) {
    if (o.wires.size() != static_cast<size_t>(s.n)) {
        raise(PLK_ERR_INVALID, "SparseH wire count does not match state-vector size");
    }
}

void apply_obs_into(Device &dev, const State &out, const State &in, const ObsNode &o) {
    if (const PauliDevice *t = o.pauli_on(dev, in.n)) {
        launch_pauli_apply(dev, out, in, *t);
        return;
    }
    if (o.kind == ObsNode::Sparse) {
        check_sparse_wires(o, in);
        csr_spmv(dev, out, in, o.csr_on(dev, in));
        return;
    }
    launch_copy(dev, out, in);
    apply_obs_general(dev, out, o);
}

void apply_obs_general(Device &dev, const State &s, const ObsNode &o) {
    switch (o.kind) {
    case ObsNode::Named:
        apply_single(dev, s, compile_op(o.name, o.wires, false, {}, {}, s.n));
        return;
    case ObsNode::Hermitian: {
        CompiledOp op;
        op.kind = OpKind::Dense;
        op.wires = o.wires;
        op.mat = o.matrix;
        apply_single(dev, s, op);
        return;
    }
    case ObsNode::Tensor:
        for (auto &t : o.terms) {
            apply_obs_general(dev, s, *t);
        }
        return;
    case ObsNode::Hamiltonian: {
        TmpState buf(s.n, s.dtype, s.device);
        TmpState tmp(s.n, s.dtype, s.device);
        launch_fill_zero(dev, buf.s);
        for (size_t t = 0; t < o.terms.size(); t++) {
            apply_obs_into(dev, tmp.s, s, *o.terms[t]);
            launch_axpy(dev, buf.s, o.coeffs[t], tmp.s);
        }
        launch_copy(dev, s, buf.s);
        PLK_HIP(hipStreamSynchronize(dev.stream));
        return;
    }
    case ObsNode::Sparse: {
        check_sparse_wires(o, s);
        TmpState tmp(s.n, s.dtype, s.device);
        csr_spmv(dev, tmp.s, s, o.csr_on(dev, s));
        launch_copy(dev, s, tmp.s);
        PLK_HIP(hipStreamSynchronize(dev.stream));
        return;
    }
    }
}

double expval_obs(Device &dev, const State &s, const ObsNode &o) {
    if (const PauliDevice *t = o.pauli_on(dev, s.n)) {
        return pauli_expval(dev, s, *t);
    }
    if (o.kind == ObsNode::Sparse) {
        // sum_r Re(conj(psi_r) (A psi)_r) without materialising A psi.
        check_sparse_wires(o, s);
        return csr_expval(dev, s, o.csr_on(dev, s));
    }
    if (o.kind == ObsNode::Hermitian) {
        // <psi|M|psi> group by group, without a copy of the state.
        return dense_expval(dev, s, o.wires, o.matrix);
    }
    TmpState tmp(s.n, s.dtype, s.device);
    launch_copy(dev, tmp.s, s);
    apply_obs_general(dev, tmp.s, o);
    const State *xs[1] = {&s};
    double ri[2];
    inner_products(dev, xs, 1, tmp.s, ri);
    return ri[0];
}

// ---------------------------------------------------------------------------
// Operation list (AdjointDiffKokkos.hpp:17-173).
// ---------------------------------------------------------------------------
struct OpsData {
    std::vector<std::string> names;
    std::vector<std::vector<double>> params;
    std::vector<std::vector<size_t>> wires;
    std::vector<bool> inverses;
    std::vector<std::vector<cd>> matrices;
    std::vector<double> angles; // the first parameter of every parametric op
    uint64_t key = 0; // hash without the matrices; full_key: with them, see ops_key
    bool dense = false;
    mutable uint64_t full_key = 0;
    mutable bool keyed = false;
    size_t num_par_ops() const { return angles.size(); }
};

// Patched gate of an op: the one-wire rotations and PhaseShift (a named gate
// ignores an explicit matrix).
int16_t patch_gate_of(const OpsData &ops, size_t i) {
    if (ops.params[i].size() != 1) {
        return BPG_NONE;
    }
    const std::string &nm = ops.names[i];
    if (nm == "RX") {
        return BPG_RX;
    }
    if (nm == "RY") {
        return BPG_RY;
    }
    if (nm == "RZ") {
        return BPG_RZ;
    }
    if (nm == "PhaseShift") {
        return BPG_PHASE;
    }
    return BPG_NONE;
}

// Hash of everything a batch plan depends on: names, wires, inverse flags,
// matrices and the parameters of gates whose angles it does not patch; the
// matrices when a batched call asks, like obs_key.
uint64_t ops_key(const OpsData &ops) {
    if (!ops.dense) {
        return ops.key;
    }
    if (!ops.keyed) {
        Hasher H;
        H.add(ops.key);
        for (const auto &matrix : ops.matrices) {
            for (const cd &m : matrix) {
                H.add(m.real());
                H.add(m.imag());
            }
        }
        ops.full_key = H.h;
        ops.keyed = true;
    }
    return ops.full_key;
}

// Adds op i to the list's hash and angles.
void note_op(OpsData &ops, Hasher &H, size_t i) {
    H.add(ops.names[i]);
    H.add(static_cast<uint64_t>(ops.wires[i].size() | (ops.inverses[i] ? size_t{1} << 40 : 0)));
    for (auto w : ops.wires[i]) {
        H.add(static_cast<uint64_t>(w));
    }
    H.add(static_cast<uint64_t>(ops.params[i].size()));
    if (patch_gate_of(ops, i) == BPG_NONE) {
        for (double v : ops.params[i]) {
            H.add(v);
        }
    }
    H.add(static_cast<uint64_t>(ops.matrices[i].size()));
    ops.dense = ops.dense || !ops.matrices[i].empty();
    if (!ops.params[i].empty()) {
        ops.angles.push_back(ops.params[i][0]);
    }
    ops.key = H.h;
}

// The whole op list, compiled (applyOperations, AdjointDiffKokkos.hpp:213-226).
std::vector<PlanOp> forward_ops(const OpsData &ops, int n) {
    std::vector<PlanOp> v;
    v.reserve(ops.names.size());
    for (size_t i = 0; i < ops.names.size(); i++) {
        PlanOp p;
        p.U = compile_op(ops.names[i], ops.wires[i], ops.inverses[i], ops.params[i],
                         ops.matrices[i], n);
        v.push_back(std::move(p));
    }
    return v;
}

// Forward plan of the whole op list. wide: as its image is built.
std::vector<Step> forward_plan(const Device &dev, std::vector<PlanOp> &&v, int n, int dtype, bool wide) {
    if (use_rtile(n, dtype, 0)) {
        std::vector<Step> steps = plan_tiles(std::move(v), n, plan_reg_bits(n, dtype, 0, 1, dev.num_cus, wide) + RT_LANE_BITS,
                                             low_bits(dtype), RT_SLOTS_MAX, false, plan_exchange(n, dtype, 1));
        split_sparse_passes(steps, n, true);
        return steps;
    }
    const int T = tile_bits_forward(n, dtype);
    if (T > 0) {
        return plan_tiles(std::move(v), n, T, low_bits(dtype));
    }
    return plan_steps(std::move(v));
}

bool is_unitary(const std::vector<cd> &M, size_t dim, double tol) {
    for (size_t a = 0; a < dim; a++) {
        for (size_t b = 0; b <= a; b++) {
            cd s = a == b ? -1.0 : 0.0;
            for (size_t r = 0; r < dim; r++) {
                s += std::conj(M[r * dim + a]) * M[r * dim + b];
            }
            if (!(std::abs(s) <= tol)) {
                return false;
            }
        }
    }
    return true;
}

// The reverse walk of AdjointDiffKokkos.hpp:432-470: U^dagger of every op
// after the last trainable one, in reverse order, each trainable op carrying
// its generator, Jacobian column and coefficient -2 s (inverse ? -1 : 1).
// StatePrep / BasisState are skipped; ops with several parameters abort.
// unitary: largest entry of U^dag U - 1 at which an explicit matrix still counts
// as unitary (a matrix that a complex64 program gives in its own precision). One
// on five wires or more counts as skew unseen: the look takes 8^m products, and
// all that it would save is that runs of gates end there.
std::vector<PlanOp> reverse_ops(const OpsData &ops, const std::vector<size_t> &tp, int n, int dtype) {
    const double unitary = dtype == PLK_C64 ? 1e-6 : 1e-12;
    const size_t n_tp = tp.size();
    std::vector<PlanOp> rev;
    size_t trainable_number = n_tp - 1;
    size_t current_param_idx = ops.num_par_ops() - 1;
    auto tp_it = tp.rbegin();
    for (long op_idx = static_cast<long>(ops.names.size()) - 1; op_idx >= 0; op_idx--) {
        const size_t o = static_cast<size_t>(op_idx);
        if (ops.params[o].size() > 1) {
            raise(PLK_ERR_INVALID,
                  "The operation is not supported using the adjoint "
                  "differentiation method");
        }
        if (ops.names[o] == "StatePrep" || ops.names[o] == "BasisState") {
            continue;
        }
        if (tp_it == tp.rend()) {
            break;
        }
        PlanOp p;
        p.U = compile_op(ops.names[o], ops.wires[o], !ops.inverses[o], ops.params[o],
                         ops.matrices[o], n);
        p.src = static_cast<int32_t>(o);
        p.adj = !ops.inverses[o];
        p.skew = !is_named_gate(ops.names[o]) && p.U.kind == OpKind::Dense &&
                 (p.U.wires.size() > 4 || !is_unitary(p.U.mat, size_t{1} << p.U.wires.size(), unitary));
        if (!ops.params[o].empty()) {
            if (current_param_idx == *tp_it) {
                p.trainable = true;
                p.G = compile_generator(ops.names[o], ops.wires[o], n);
                p.coef = -2.0 * p.G.scale * (ops.inverses[o] ? -1.0 : 1.0);
                p.col = static_cast<int>(trainable_number);
                trainable_number--;
                ++tp_it;
            }
            current_param_idx--;
        }
        rev.push_back(std::move(p));
    }
    return rev;
}

// ---------------------------------------------------------------------------
// Adjoint Jacobian (AdjointDiffKokkos.hpp:404-478).
//
// The reverse walk over the operations, the trainable-parameter bookkeeping
// and the early stop follow the reference line by line; the per-operation
// work (mu copy, U^dagger on lambda, generator on mu, n_obs inner products,
// U^dagger on every H lambda) is replaced by fused passes.
// ---------------------------------------------------------------------------

// One launch of a register-tile pass or of a single-op step: its observables
// j0 .. j0 + width and where its FP64 partials start.
struct PartLaunch {
    size_t j0 = 0;
    int width = 0;
    RtLaunch rt{};
    StepLaunch step{};
    size_t offset = 0; // doubles from the device's partials buffer
};

// The launches of a reverse plan and the reductions of their partials. Every
// pass keeps its partials until a flush, which forms all Jacobian entries
// since the last one in one launch (a launch per pass costs small circuits
// as much as the passes themselves).
struct SweepParts {
    std::vector<std::vector<PartLaunch>> steps;
    struct Flush {
        size_t step;         // after this step
        size_t first, count; // entries
    };
    std::vector<Flush> flushes;
    size_t doubles = 0;
};

constexpr size_t kPartialsMax = size_t{1} << 26; // doubles kept between flushes

// Places the partials of every launch and fills img.entries.
SweepParts place_partials(Device &dev, const std::vector<Step> &steps, PlanImage &img, const State &s,
                          size_t n_obs, bool alt) {
    SweepParts sp;
    sp.steps.resize(steps.size());
    if (n_obs > static_cast<size_t>(SEG_NJMAX)) {
        img.slabs.clear(); // several chunks read phi before the last one writes it
    }
    size_t used = 0, first = 0;
    auto flush = [&](size_t i) {
        if (img.entries.size() > first) {
            sp.flushes.push_back({i, first, img.entries.size() - first});
            first = img.entries.size();
        }
        used = 0;
    };
    auto take = [&](size_t i, PartLaunch &pl, size_t doubles) {
        if (used + doubles > kPartialsMax && i > 0 && used > 0 && sp.steps[i].empty()) {
            flush(i - 1);
        }
        pl.offset = used;
        used += doubles;
        sp.doubles = std::max(sp.doubles, used);
    };
    auto entry = [](const PartLaunch &pl, int blocks, int col) {
        RtEntry e{};
        e.base = pl.offset;
        e.row[0] = e.row[1] = e.row[2] = -1;
        e.blocks = blocks;
        e.col = col;
        e.j0 = static_cast<int32_t>(pl.j0);
        e.width = pl.width;
        return e;
    };
    for (size_t i = 0; i < steps.size(); i++) {
        const Step &st = steps[i];
        if (st.tiled && st.pass.rt) {
            // The chunks (balanced: widths nj and nj - 1, wider first) run side
            // by side in one launch, up to RT_OBS_MAX states, when lambda has a
            // second buffer.
            const std::vector<int> sizes = chunk_sizes(n_obs, rtile_chunk(s.dtype, s.n, dev.num_cus));
            size_t j0 = 0;
            for (size_t ci = 0; ci < sizes.size();) {
                PartLaunch pl;
                RtLaunch &L = pl.rt;
                L = img.progs[i].L;
                L.nj = sizes[0];
                L.nc = 1;
                L.nbig = sizes[ci] == L.nj ? 1 : 0;
                pl.width = sizes[ci];
                while (alt && ci + L.nc < sizes.size() && pl.width + sizes[ci + L.nc] <= RT_OBS_MAX) {
                    pl.width += sizes[ci + L.nc];
                    L.nbig += sizes[ci + L.nc] == L.nj ? 1 : 0;
                    L.nc++;
                }
                pl.j0 = j0;
                L.write_phi = j0 + pl.width == n_obs ? 1 : 0;
                const int blocks = rtile_blocks(dev, s.dtype, L);
                take(i, pl, static_cast<size_t>(L.nslots) * pl.width * blocks);
                for (const RtTerm &t : img.progs[i].terms) {
                    RtEntry e = entry(pl, blocks, t.col);
                    for (int k = 0; k < 3; k++) {
                        e.row[k] = t.slot[k] < 0 ? -1 : t.slot[k] * pl.width;
                        e.m[k] = t.m[k];
                    }
                    img.entries.push_back(e);
                }
                j0 += pl.width;
                ci += L.nc;
                sp.steps[i].push_back(pl);
            }
        } else if (const SlabGroup *g = slab_of(img, i)) {
            // All steps of the launch keep their partials until it has run.
            const StepMeta &m = img.singles[i];
            const size_t slabs = size_t{1} << (g->L.n - g->L.S);
            if (i == g->first && used + g->count * n_obs * slabs > kPartialsMax && used > 0) {
                flush(i - 1);
            }
            PartLaunch pl;
            pl.step = m.L;
            pl.step.nj = static_cast<int>(n_obs);
            pl.width = static_cast<int>(n_obs);
            if (m.L.trainable) {
                pl.offset = used;
                used += n_obs * slabs;
                sp.doubles = std::max(sp.doubles, used);
                const uint64_t part = pl.offset;
                std::memcpy(img.mats.data() + g->off + (i - g->first) * sizeof(SlabStep) + offsetof(SlabStep, part),
                            &part, sizeof part);
                RtEntry e = entry(pl, static_cast<int>(slabs), m.col);
                e.row[0] = 0;
                e.m[0] = m.coef;
                img.entries.push_back(e);
            }
            sp.steps[i].push_back(pl);
        } else if (!st.fused && !st.tiled && img.singles[i].ok) {
            const StepMeta &m = img.singles[i];
            size_t j0 = 0;
            for (int nj : chunk_sizes(n_obs, SEG_NJMAX)) {
                PartLaunch pl;
                pl.step = m.L;
                pl.step.nj = nj;
                pl.j0 = j0;
                pl.width = nj;
                pl.step.write_phi = (j0 + nj == n_obs) ? 1 : 0;
                if (m.L.trainable) {
                    const int blocks = step_blocks(dev, pl.step);
                    take(i, pl, static_cast<size_t>(nj) * blocks);
                    RtEntry e = entry(pl, blocks, m.col);
                    e.row[0] = 0;
                    e.m[0] = m.coef;
                    img.entries.push_back(e);
                }
                j0 += nj;
                sp.steps[i].push_back(pl);
            }
        }
    }
    if (!steps.empty()) {
        flush(steps.size() - 1);
    }
    return sp;
}

// Launches reverse step i (a fused segment, register-tile or LDS-tile pass
// over lambda and every H_j lambda, with its Jacobian reductions); returns
// false for a single op, which the caller runs.
// The adjoint's lambda. Register-tile passes run their observable chunks
// side by side, all reading cur, and write the updated lambda to alt; the
// two then swap. Without alt (one chunk) they update cur in place.
struct PhiPair {
    State cur, alt;
};

bool enqueue_reverse_step(Device &dev, PhiPair &phi, void *const *hptr, size_t n_obs,
                          size_t n_tp, const Step &st, const PlanImage &img, size_t i,
                          const PlanPlace &pl, const SweepParts &parts, double *d_jac) {
    const State &lambda = phi.cur;
    if (const SlabGroup *g = slab_of(img, i)) {
        if (g->first == i) {
            SlabLaunch L = g->L;
            L.nj = static_cast<int>(n_obs);
            launch_slab_steps(dev, lambda, hptr, pl.mats, pl.mats + g->off, L, dev.parts);
        }
        return true;
    }
    if (st.fused) {
        const SegMeta &m = img.metas[i];
        const int njmax = std::min(SEG_NJMAX, seg_max_nj(lambda.dtype, m.L.K));
        size_t j0 = 0;
        while (j0 < n_obs) {
            const size_t left = n_obs - j0;
            int nj = 1;
            for (int c : {8, 4, 2, 1}) {
                if (c <= njmax && static_cast<size_t>(c) <= left) {
                    nj = c;
                    break;
                }
            }
            SegLaunch L = m.L;
            L.nj = nj;
            L.write_phi = (j0 + nj == n_obs) ? 1 : 0;
            const int grid = launch_segment(dev, lambda, hptr + j0, pl.ops + m.first, L);
            if (L.nslots > 0) {
                launch_segment_reduce(dev, grid, L.nslots, nj, static_cast<int>(j0), m.cols,
                                      m.coefs, d_jac, static_cast<int>(n_tp));
            }
            j0 += nj;
        }
        return true;
    }
    if (st.tiled && st.pass.rt) {
        for (const PartLaunch &l : parts.steps[i]) {
            const bool swap = l.rt.write_phi && phi.alt.d != nullptr;
            launch_rtile(dev, phi.cur, swap ? &phi.alt : nullptr, hptr + l.j0, pl.rt + img.progs[i].off, l.rt,
                         dev.parts + l.offset);
            if (swap) {
                std::swap(phi.cur, phi.alt);
            }
        }
        return true;
    }
    if (!st.fused && !st.tiled && img.singles[i].ok) {
        for (const PartLaunch &l : parts.steps[i]) {
            launch_step(dev, lambda, hptr + l.j0, pl.mats + img.singles[i].off, l.step, dev.parts + l.offset);
        }
        return true;
    }
    if (st.tiled) {
        const SegMeta &m = img.metas[i];
        size_t j0 = 0;
        for (int nj : chunk_sizes(n_obs, tile_max_nj(lambda.dtype, m.TL.T))) {
            TileLaunch TL = m.TL;
            TL.nj = nj;
            TL.write_phi = (j0 + nj == n_obs) ? 1 : 0;
            const int grid = launch_tile(dev, lambda, hptr + j0, pl.bundles + m.first_bundle,
                                         pl.ops, TL);
            if (TL.nslots > 0) {
                launch_tile_reduce(dev, grid, TL.nslots, nj, static_cast<int>(j0),
                                   st.pass.cols.data(), st.pass.coefs.data(), d_jac,
                                   static_cast<int>(n_tp));
            }
            j0 += nj;
        }
        return true;
    }
    return false;
}

// Forms the Jacobian entries whose partials end with step i.
void enqueue_flush(Device &dev, const SweepParts &parts, const PlanPlace &pl, size_t i, size_t n_obs,
                   size_t n_tp, double *d_jac) {
    for (const auto &f : parts.flushes) {
        if (f.step == i) {
            launch_rtile_entries(dev, dev.parts, pl.entries + f.first, static_cast<int>(f.count),
                                 static_cast<int>(n_obs), d_jac, static_cast<int>(n_tp));
        }
    }
}

// A captured sweep: copy of the input state, forward passes, observables,
// Jacobian zero fill and reverse passes of one circuit structure, replayed
// with a fresh upload of the plan and Pauli tables (angles and coefficients
// live there). The graph owns every buffer its kernels touch except the
// input state and the device's partials buffer (checked before each replay).
struct SweepGraph {
    uint64_t key = 0;
    int device = -1;
    hipStream_t stream = nullptr;
    const void *ref = nullptr;
    std::vector<unsigned char> sig;
    std::unique_ptr<TmpState> lambda, lambda2; // lambda2: second buffer of PhiPair (or none)
    std::vector<std::unique_ptr<TmpState>> H;
    std::vector<void *> hptr;
    void *tables = nullptr;
    size_t fwd_bytes = 0, rev_bytes = 0;
    double *jac = nullptr;
    double *red = nullptr, *parts = nullptr;
    hipGraphExec_t exec = nullptr;
    ~SweepGraph() {
        (void)hipSetDevice(device);
        (void)hipStreamSynchronize(stream);
        if (exec) {
            (void)hipGraphExecDestroy(exec);
        }
        if (tables) {
            (void)hipFree(tables);
        }
        if (jac) {
            (void)hipFree(jac);
        }
    }
};

// Up to 21 qubits launches are short enough for their host cost to show (20
// qubits, 360 single-op steps: 4.5 ms replayed, 5.9 ms launched one by one).
constexpr int kGraphMaxQubits = 21;
constexpr size_t kGraphsPerDevice = 128;
constexpr size_t kGraphBytesPerDevice = size_t{4} << 30; // states held by graphs

std::map<int, std::vector<std::unique_ptr<SweepGraph>>> &sweep_graphs() {
    static std::map<int, std::vector<std::unique_ptr<SweepGraph>>> g; // released with the process
    return g;
}

// Structures seen once (a capture pays off from the second call on).
std::map<int, std::map<uint64_t, int>> &sweep_seen() {
    static std::map<int, std::map<uint64_t, int>> seen;
    return seen;
}

size_t graph_bytes(const SweepGraph &g) {
    return (1 + g.H.size() + (g.lambda2 ? 1 : 0)) * g.lambda->s.bytes();
}

// Whether the reverse plan runs register-tile chunks side by side, which
// needs lambda in two buffers.
bool needs_alt(const Device &dev, const std::vector<Step> &steps, size_t n_obs, int dtype, int n) {
    if (n_obs <= static_cast<size_t>(rtile_chunk(dtype, n, dev.num_cus))) {
        return false;
    }
    for (const auto &st : steps) {
        if (st.tiled && st.pass.rt) {
            return true;
        }
    }
    return false;
}

// Everything but the angles: op names / wires / inverse flags / parameter
// counts / matrix sizes, the trainable set, sizes and flags.
uint64_t sweep_key(const State &ref, const OpsData &ops, const std::vector<size_t> &tp,
                   size_t n_obs, bool apply_ops) {
    Hasher H;
    H.add(static_cast<uint64_t>(ref.n));
    H.add(static_cast<uint64_t>(ref.dtype));
    H.add(static_cast<uint64_t>(n_obs));
    H.add(static_cast<uint64_t>(apply_ops ? 1 : 0));
    H.add(static_cast<uint64_t>(ops.names.size()));
    for (size_t i = 0; i < ops.names.size(); i++) {
        H.add(ops.names[i]);
        H.add(static_cast<uint64_t>(ops.wires[i].size() | (ops.inverses[i] ? size_t{1} << 40 : 0)));
        for (auto w : ops.wires[i]) {
            H.add(static_cast<uint64_t>(w));
        }
        H.add(static_cast<uint64_t>(ops.params[i].size()));
        H.add(static_cast<uint64_t>(ops.matrices[i].size()));
    }
    H.add(static_cast<uint64_t>(tp.size()));
    for (auto t : tp) {
        H.add(static_cast<uint64_t>(t));
    }
    return H.h;
}

// Stream capture with profiling scopes off; always ends the capture.
struct CaptureGuard {
    hipStream_t stream;
    bool open = true;
    explicit CaptureGuard(hipStream_t s) : stream(s) {
        set_capturing(true);
        PLK_HIP(hipStreamBeginCapture(stream, hipStreamCaptureModeRelaxed));
    }
    hipGraph_t end() {
        hipGraph_t g = nullptr;
        open = false;
        set_capturing(false);
        PLK_HIP(hipStreamEndCapture(stream, &g));
        return g;
    }
    ~CaptureGuard() {
        if (open) {
            hipGraph_t g = nullptr;
            set_capturing(false);
            if (hipStreamEndCapture(stream, &g) == hipSuccess && g) {
                (void)hipGraphDestroy(g);
            }
        }
    }
};

// Whether a plan holds a single-op step outside the step kernels (those
// synchronise with the host, so the plan cannot be captured).
bool steps_have_single(const std::vector<Step> &steps, int n) {
    for (const auto &st : steps) {
        if (!st.fused && !st.tiled && !step_kernel_ok(st.single, n)) {
            return true;
        }
    }
    return false;
}

// The launches of a reverse plan and where their partials lie: the entries
// that a replay copies have to match the launches it replays.
void append_signature(const SweepParts &parts, std::vector<unsigned char> &sig) {
    auto put = [&](uint64_t v) {
        const auto *b = reinterpret_cast<const unsigned char *>(&v);
        sig.insert(sig.end(), b, b + sizeof v);
    };
    for (const auto &step : parts.steps) {
        put(step.size());
        for (const PartLaunch &l : step) {
            for (const uint64_t v : {static_cast<uint64_t>(l.j0), static_cast<uint64_t>(l.width),
                                     static_cast<uint64_t>(l.offset), static_cast<uint64_t>(l.rt.nj),
                                     static_cast<uint64_t>(l.rt.nc), static_cast<uint64_t>(l.rt.nbig),
                                     static_cast<uint64_t>(l.rt.write_phi), static_cast<uint64_t>(l.step.nj),
                                     static_cast<uint64_t>(l.step.write_phi)}) {
                put(v);
            }
        }
    }
    for (const auto &f : parts.flushes) {
        put(f.step);
        put(f.first);
        put(f.count);
    }
    put(parts.doubles);
}

// ---------------------------------------------------------------------------
// Whole circuits in one launch (kernels_sweep.hip): one workgroup per
// observable runs every pass of the circuit.
// ---------------------------------------------------------------------------
// Up to 12 qubits the launch beats a launch per pass (12 qubits, 12
// observables, complex128: 0.36 against 0.53 ms a Jacobian), but for observables of
// many words and lists of a few operations (sweep_takes_words, sweep_pays_forward).
// PLK_SWEEP=0 turns it off.
constexpr int kSweepQubits = 12;

bool sweep_serves(const State &s) {
    return s.n <= kSweepQubits && env_int("PLK_SWEEP", 1) != 0 && env_int("PLK_RTILE", -1) != 0;
}

// Every op fits a register-tile pass.
bool sweep_takes(std::vector<PlanOp> &ops) {
    for (auto &p : ops) {
        if (p.U.kind == OpKind::Identity && !p.trainable) {
            continue;
        }
        prepare(p);
        if (!fusable(p)) {
            return false;
        }
    }
    return true;
}

// Host tables of a whole-circuit launch.
struct SweepTables {
    std::vector<SweepPass> passes;
    std::vector<SweepEntry> entries;
    std::vector<SweepTerm> terms;
    std::vector<unsigned char> blob;

    // Batch plans (patched): the runs with angles.
    std::vector<BatchRun> runs;
    std::vector<BatchGate> gates;
    std::vector<double> consts; // 2x2 complex matrices

    // Plans ops into passes whose tiles hold the lowest L bits; returns the
    // first and the number of them.
    std::pair<int, int> add(std::vector<PlanOp> &&ops, int n, int dtype, int L = 0, bool patched = false) {
        const int R = sweep_reg_bits(dtype), T = R + RT_LANE_BITS;
        const int first = static_cast<int>(passes.size());
        double norm = 1.0;
        for (Step &st : plan_tiles(std::move(ops), n, T, L, RT_SLOTS_MAX, false)) {
            if (!st.tiled) {
                raise(PLK_ERR_UNSUPPORTED,
                      "batched circuits support dense gates and generators on at most two wires");
            }
            for (int b = n; static_cast<int>(st.pass.tb.size()) < T; b++) {
                st.pass.tb.push_back(b); // idle bits of a state smaller than a tile
            }
            const RtProgram pr = dtype == PLK_C64 ? build_rt_program<float>(st.pass, n, R, keep_bits(dtype), blob, norm, patched)
                                                  : build_rt_program<double>(st.pass, n, R, keep_bits(dtype), blob, norm, patched);
            SweepPass P{};
            P.prog = static_cast<int64_t>(pr.off);
            P.T = T;
            P.ninstr = pr.L.ninstr;
            P.nslots = pr.L.nslots;
            P.entry_first = static_cast<int32_t>(entries.size());
            P.entry_count = static_cast<int32_t>(pr.terms.size());
            for (const RtPatch &pt : pr.patches) {
                BatchRun r{};
                r.ins = P.prog + static_cast<int64_t>(pt.ins);
                r.first = static_cast<int32_t>(gates.size());
                r.entry = pt.term < 0 ? -1 : P.entry_first + pt.term;
                r.ukind = pt.ukind;
                r.parts = pt.parts;
                for (const RunGate &g : st.pass.ops[pt.op].gates) {
                    gates.push_back(g.g);
                    if (g.g.gate == BPG_CONST) {
                        gates.back().param = static_cast<int32_t>(consts.size() / 8);
                        for (const cd &m : g.mat) {
                            consts.push_back(m.real());
                            consts.push_back(m.imag());
                        }
                    }
                }
                r.count = static_cast<int32_t>(gates.size()) - r.first;
                runs.push_back(r);
            }
            std::copy(pr.L.tb, pr.L.tb + RT_TMAX, P.tb);
            std::copy(pr.L.reg_in, pr.L.reg_in + RT_RMAX, P.reg_in);
            std::copy(pr.L.reg_out, pr.L.reg_out + RT_RMAX, P.reg_out);
            std::copy(pr.L.lane_in, pr.L.lane_in + RT_LANE_BITS, P.lane_in);
            std::copy(pr.L.lane_out, pr.L.lane_out + RT_LANE_BITS, P.lane_out);
            passes.push_back(P);
            for (const RtTerm &t : pr.terms) {
                entries.push_back({t.col, {t.slot[0], t.slot[1], t.slot[2]}, {t.m[0], t.m[1], t.m[2]}});
            }
        }
        return {first, static_cast<int>(passes.size()) - first};
    }
};

int sweep_waves(int n, int dtype) {
    const int T = sweep_reg_bits(dtype) + RT_LANE_BITS;
    return n > T ? std::min(kSweepWaves, 1 << (n - T)) : 1;
}

// Uploads the tables and the jobs (one copy) and launches; waits for the
// stream, which has then read the host image.
void run_sweep(Device &dev, int dtype, int n, const SweepTables &t, const std::vector<SweepJob> &jobs,
               std::vector<double> *jac, const double *d_jac) {
    auto up = [](size_t x) { return (x + 255) & ~size_t{255}; };
    const size_t o_pass = up(jobs.size() * sizeof(SweepJob));
    const size_t o_ent = o_pass + up(t.passes.size() * sizeof(SweepPass));
    const size_t o_term = o_ent + up(t.entries.size() * sizeof(SweepEntry));
    const size_t o_blob = o_term + up(t.terms.size() * sizeof(SweepTerm));
    std::vector<unsigned char> host(o_blob + up(t.blob.size()));
    auto put = [&](size_t off, const void *src, size_t bytes) {
        if (bytes) {
            std::memcpy(host.data() + off, src, bytes);
        }
    };
    put(0, jobs.data(), jobs.size() * sizeof(SweepJob));
    put(o_pass, t.passes.data(), t.passes.size() * sizeof(SweepPass));
    put(o_ent, t.entries.data(), t.entries.size() * sizeof(SweepEntry));
    put(o_term, t.terms.data(), t.terms.size() * sizeof(SweepTerm));
    put(o_blob, t.blob.data(), t.blob.size());
    auto *d = static_cast<unsigned char *>(arena_alloc(dev, host.size()));
    PLK_HIP(hipMemcpyAsync(d, host.data(), host.size(), hipMemcpyHostToDevice, dev.stream));
    SweepArgs A;
    A.jobs = reinterpret_cast<const SweepJob *>(d);
    A.passes = reinterpret_cast<const SweepPass *>(d + o_pass);
    A.entries = reinterpret_cast<const SweepEntry *>(d + o_ent);
    A.terms = reinterpret_cast<const SweepTerm *>(d + o_term);
    A.blob = d + o_blob;
    launch_sweep(dev, dtype, A, static_cast<int>(jobs.size()), sweep_waves(n, dtype));
    if (jac != nullptr && !jac->empty()) {
        PLK_HIP(hipMemcpyAsync(jac->data(), d_jac, jac->size() * sizeof(double), hipMemcpyDeviceToHost,
                               dev.stream));
    }
    PLK_HIP(hipStreamSynchronize(dev.stream));
}

// Op lists that run whole in one launch. A handful of operations is one or two
// launches in the general path too, with less to plan and upload (general /
// whole: 5 qubits complex128 1 op 14.7 / 16.9 us, 4 ops 18.2 / 18.4, 8 ops 21 / 19;
// complex64 4 ops 17.9 / 19.3, 8 one-wire ops 22.1 / 21.4; states of at most three
// wires, one register segment: 8 ops 18.0 / 18.9).
bool sweep_pays_forward(const State &s, size_t ops) {
    return ops > (s.n <= SEG_KMAX ? 8u : s.dtype == PLK_C64 ? 6u : 4u);
}

void sweep_forward(Device &dev, const State &s, std::vector<PlanOp> &&ops) {
    SweepTables t;
    SweepJob J{};
    J.n = s.n;
    std::tie(J.fwd_first, J.fwd_count) = t.add(std::move(ops), s.n, s.dtype);
    J.ref = J.phi = s.d;
    run_sweep(dev, s.dtype, s.n, t, {J}, nullptr, nullptr);
}

// Pauli words of an observable, at least, without expanding it.
size_t least_words(const ObsNode &o) {
    return o.kind == ObsNode::Hamiltonian ? o.terms.size() : 1;
}

// Whether the whole-circuit launch forms H lambda fast enough: there one
// workgroup walks every word of an observable for each of its amplitudes (0.036
// us a word and amplitude of a thread more than the general path, whose launch
// has the whole chip), where the general path has a launch and an upload for each
// observable (6 us and 0.2 to 0.3 us a word). One observable, one layer, whole / general:
// 12 qubits complex128 64 words 154 / 159 us, 128 words 191 / 189, 600 words
// 547 / 420; 12 qubits complex64 32 words 140 / 137, 600 words 743 / 425; 10 qubits
// complex64 64 words 144 / 148, 128 words 196 / 181. Four observables of 600 words
// each, 12 qubits complex128: 889 / 1291. Below nine qubits the general path has no
// register-tile passes: 8 qubits complex128, 600 words 361 / 410, 1500 words 821 / 763.
bool sweep_takes_words(const std::vector<std::shared_ptr<const ObsNode>> &obs, int n, int dtype) {
    const size_t threads = static_cast<size_t>(64) * sweep_waves(n, dtype);
    const size_t each = std::max<size_t>(1, (size_t{1} << n) / threads);
    size_t most = 0, all = 0;
    for (const auto &o : obs) {
        const size_t words = least_words(*o);
        most = std::max(most, words);
        all += 6 * words + 165;
    }
    return most * each <= (n < 9 ? 2500 : 800) + all - (6 * most + 165);
}

// The Jacobian by one workgroup per observable; false when an op or an
// observable needs the general path. rev: the reverse walk's ops.
bool sweep_jacobian(Device &dev, const State &ref, const std::vector<std::shared_ptr<const ObsNode>> &obs,
                    const OpsData &ops, std::vector<PlanOp> &rev, size_t n_tp, bool apply_ops, double *jac) {
    const int n = ref.n;
    if (!sweep_serves(ref) || !sweep_takes_words(obs, n, ref.dtype) || !sweep_takes(rev)) {
        return false;
    }
    SweepTables t;
    std::vector<SweepJob> jobs(obs.size());
    for (size_t j = 0; j < obs.size(); j++) {
        std::vector<PauliTerm> terms;
        if (!to_pauli(*obs[j], n, terms)) {
            return false;
        }
        jobs[j].term_first = static_cast<int32_t>(t.terms.size());
        jobs[j].term_count = static_cast<int32_t>(terms.size());
        for (const auto &p : terms) {
            t.terms.push_back({static_cast<uint32_t>(p.x), static_cast<uint32_t>(p.zy), p.coeff.real(),
                               p.coeff.imag()});
        }
    }
    std::vector<PlanOp> fwd;
    if (apply_ops) {
        fwd = forward_ops(ops, n);
        if (!sweep_takes(fwd)) {
            return false;
        }
    }
    const std::pair<int, int> f = t.add(std::move(fwd), n, ref.dtype);
    const std::pair<int, int> r = t.add(std::move(rev), n, ref.dtype);
    const size_t bytes = (ref.bytes() + 255) & ~size_t{255};
    auto *scratch = static_cast<unsigned char *>(arena_alloc(dev, 2 * bytes * obs.size()));
    double *d_jac = ensure_jac(dev, obs.size() * n_tp);
    for (size_t j = 0; j < obs.size(); j++) {
        SweepJob &J = jobs[j];
        J.n = n;
        std::tie(J.fwd_first, J.fwd_count) = f;
        std::tie(J.rev_first, J.rev_count) = r;
        J.jac_len = static_cast<int32_t>(n_tp);
        J.ref = ref.d;
        J.phi = scratch + 2 * j * bytes;
        J.h = scratch + (2 * j + 1) * bytes;
        J.jac = d_jac + j * n_tp;
    }
    std::vector<double> out(obs.size() * n_tp);
    run_sweep(dev, ref.dtype, n, t, jobs, &out, d_jac);
    std::copy(out.begin(), out.end(), jac);
    return true;
}

void adjoint_jacobian(const State &ref, const std::vector<std::shared_ptr<const ObsNode>> &obs,
                      const OpsData &ops, const std::vector<size_t> &tp, bool apply_ops,
                      double *jac) {
    if (tp.empty()) {
        raise(PLK_ERR_INVALID, "No trainable parameters provided.");
    }
    const size_t n_obs = obs.size();
    const size_t n_tp = tp.size();
    std::fill(jac, jac + n_obs * n_tp, 0.0);
    Device &dev = dev_of(ref);
    const int n = ref.n;

    // Reverse plan first: it validates the op list before any device work.
    std::unique_ptr<HostScope> plan_scope = std::make_unique<HostScope>("host_adjoint_plan");
    std::vector<PlanOp> rev = reverse_ops(ops, tp, n, ref.dtype);
    if (n_obs == 0) {
        return;
    }
    if (sweep_jacobian(dev, ref, obs, ops, rev, n_tp, apply_ops, jac)) {
        return;
    }
    const int nj = sweep_chunk(ref.dtype, n, n_obs, dev.num_cus);
    const bool rt = use_rtile(n, ref.dtype, nj);
    const int T_adj = rt ? plan_reg_bits(n, ref.dtype, nj, chunk_sizes(n_obs, nj).size(), dev.num_cus, false) + RT_LANE_BITS : tile_bits_adjoint(n, ref.dtype);
    std::vector<Step> steps =
        rt ? plan_tiles(std::move(rev), n, T_adj, low_bits(ref.dtype), RT_SLOTS_MAX, false,
                        plan_exchange(n, ref.dtype, n_obs + 1))
           : T_adj > 0 ? plan_tiles(std::move(rev), n, T_adj, low_bits(ref.dtype))
                       : plan_steps(std::move(rev));
    if (rt) {
        split_sparse_passes(steps, n, false);
    }
    const std::vector<Step> fwd = apply_ops ? forward_plan(dev, forward_ops(ops, n), n, ref.dtype, false) : std::vector<Step>{};
    const PlanImage img_f = build_image(fwd, ref, false);
    PlanImage img_r = build_image(steps, ref, false);
    const bool alt = needs_alt(dev, steps, n_obs, ref.dtype, n);
    const SweepParts parts = place_partials(dev, steps, img_r, ref, n_obs, alt);
    plan_scope.reset();

    // Small circuits run as a replayed HIP graph: their sweeps are hundreds
    // of launches of a few microseconds each.
    // Observables enter the graph as Pauli tables copied with the plan
    // tables, so circuits that differ only in angles or in observable
    // coefficients share one graph.
    struct PauliImg {
        std::vector<unsigned char> bytes;
        size_t toff = 0;
        int ngroups = 0;
    };
    std::vector<PauliImg> pimg;
    bool graph = n <= kGraphMaxQubits && env_int("PLK_GRAPH", 1) != 0 &&
                 (2 + n_obs) * ref.bytes() <= kGraphBytesPerDevice && // one graph alone stays in the bound
                 !steps_have_single(steps, n) && !steps_have_single(fwd, n);
    for (size_t j = 0; graph && j < n_obs; j++) {
        std::vector<PauliTerm> terms;
        graph = to_pauli(*obs[j], n, terms);
        PauliImg pi;
        if (graph) {
            pi.bytes = pauli_image(terms, pi.toff, pi.ngroups);
        }
        pimg.push_back(std::move(pi));
    }
    const uint64_t key = graph ? sweep_key(ref, ops, tp, n_obs, apply_ops) : 0;
    if (graph) {
        auto &seen = sweep_seen()[dev.id];
        if (seen.size() > 65536) {
            seen.clear();
        }
        graph = ++seen[key] >= 2;
    }
    if (graph) {
        std::unique_ptr<HostScope> phase = std::make_unique<HostScope>("host_adjoint_graph");
        std::vector<unsigned char> sig;
        append_signature(img_f, sig);
        append_signature(img_r, sig);
        append_signature(parts, sig);
        size_t pauli_bytes = 0;
        for (const auto &pi : pimg) {
            const uint64_t f[3] = {pi.bytes.size(), pi.toff, static_cast<uint64_t>(pi.ngroups)};
            const auto *b = reinterpret_cast<const unsigned char *>(f);
            sig.insert(sig.end(), b, b + sizeof f);
            pauli_bytes += (pi.bytes.size() + 255) & ~size_t{255};
        }
        auto &list = sweep_graphs()[dev.id];
        SweepGraph *g = nullptr;
        for (auto it = list.begin(); it != list.end(); ++it) {
            SweepGraph &c = **it;
            const bool same = c.key == key && c.ref == ref.d;
            if (same) {
                if (c.sig != sig || c.red != dev.red || c.parts != dev.parts) {
                    list.erase(it); // stale layout or partials buffer: capture again
                } else {
                    std::rotate(it, it + 1, list.end()); // most recently used last
                    g = list.back().get();
                }
                break;
            }
        }
        if (g == nullptr) {
            // Least recently used first in the list: evict from the front.
            size_t held = 0;
            for (const auto &c : list) {
                held += graph_bytes(*c);
            }
            const size_t need = (2 + n_obs) * ref.bytes();
            while (!list.empty() &&
                   (list.size() >= kGraphsPerDevice || held + need > kGraphBytesPerDevice)) {
                held -= graph_bytes(*list.front());
                list.erase(list.begin());
            }
            auto ng = std::make_unique<SweepGraph>();
            ng->key = key;
            ng->device = dev.id;
            ng->stream = dev.stream;
            ng->ref = ref.d;
            ng->sig = sig;
            ng->lambda = std::make_unique<TmpState>(n, ref.dtype, ref.device);
            if (alt) {
                ng->lambda2 = std::make_unique<TmpState>(n, ref.dtype, ref.device);
            }
            for (size_t j = 0; j < n_obs; j++) {
                ng->H.push_back(std::make_unique<TmpState>(n, ref.dtype, ref.device));
                ng->hptr.push_back(ng->H.back()->s.d);
            }
            ng->fwd_bytes = image_bytes(img_f);
            ng->rev_bytes = image_bytes(img_r);
            ng->tables = dev_malloc(dev.id, ng->fwd_bytes + ng->rev_bytes + pauli_bytes + 256,
                                    "graph tables");
            ng->jac = static_cast<double *>(dev_malloc(dev.id, sizeof(double) * n_obs * n_tp, "graph Jacobian"));
            // The launchers grow the partials buffer on demand, which would
            // synchronise inside the capture: size it for any pass first.
            ensure_red(dev, static_cast<size_t>(dev.num_cus) * 32 * TILE_PMAX * SEG_NJMAX, 256);
            ensure_parts(dev, parts.doubles);
            auto *tb = static_cast<unsigned char *>(ng->tables);
            // Addresses only: the tables are copied before every replay.
            const PlanPlace pf = place_addresses(img_f, tb);
            const PlanPlace pr = place_addresses(img_r, tb + ng->fwd_bytes);
            {
                CaptureGuard cap(dev.stream);
                const State &lam = ng->lambda->s;
                launch_copy(dev, lam, ref);
                enqueue_forward(dev, lam, fwd, img_f, pf);
                unsigned char *pt = tb + ng->fwd_bytes + ng->rev_bytes;
                for (size_t j = 0; j < n_obs; j++) {
                    launch_pauli_apply_at(dev, ng->H[j]->s, lam, pt, pimg[j].toff, pimg[j].ngroups);
                    pt += (pimg[j].bytes.size() + 255) & ~size_t{255};
                }
                launch_fill_zero_doubles(dev, ng->jac, n_obs * n_tp);
                PhiPair phi{lam, ng->lambda2 ? ng->lambda2->s : State{}};
                for (size_t i = 0; i < steps.size(); i++) {
                    enqueue_reverse_step(dev, phi, ng->hptr.data(), n_obs, n_tp, steps[i], img_r,
                                         i, pr, parts, ng->jac);
                    enqueue_flush(dev, parts, pr, i, n_obs, n_tp, ng->jac);
                }
                hipGraph_t graph_def = cap.end();
                const hipError_t e = hipGraphInstantiate(&ng->exec, graph_def, nullptr, nullptr, 0);
                (void)hipGraphDestroy(graph_def);
                PLK_HIP(e);
            }
            ng->red = dev.red;
            ng->parts = dev.parts;
            list.push_back(std::move(ng));
            g = list.back().get();
        }
        auto *tb = static_cast<unsigned char *>(g->tables);
        copy_image(dev, img_f, tb);
        copy_image(dev, img_r, tb + g->fwd_bytes);
        unsigned char *pt = tb + g->fwd_bytes + g->rev_bytes;
        for (const auto &pi : pimg) {
            if (!pi.bytes.empty()) {
                PLK_HIP(hipMemcpyAsync(pt, pi.bytes.data(), pi.bytes.size(), hipMemcpyHostToDevice,
                                       dev.stream));
            }
            pt += (pi.bytes.size() + 255) & ~size_t{255};
        }
        PLK_HIP(hipGraphLaunch(g->exec, dev.stream));
        PLK_HIP(hipMemcpyAsync(jac, g->jac, sizeof(double) * n_obs * n_tp, hipMemcpyDeviceToHost,
                               dev.stream));
        // Also keeps the host images alive until their copies have run.
        PLK_HIP(hipStreamSynchronize(dev.stream));
        return;
    }

    TmpState lambda(n, ref.dtype, ref.device);
    launch_copy(dev, lambda.s, ref);
    if (apply_ops) {
        enqueue_forward(dev, lambda.s, fwd, img_f, place_in_arena(dev, img_f));
    }
    std::vector<std::unique_ptr<TmpState>> H;
    for (size_t j = 0; j < n_obs; j++) {
        H.push_back(std::make_unique<TmpState>(n, ref.dtype, ref.device));
        apply_obs_into(dev, H.back()->s, lambda.s, *obs[j]);
    }
    std::vector<void *> hptr(n_obs);
    std::vector<const State *> hstate(n_obs);
    for (size_t j = 0; j < n_obs; j++) {
        hptr[j] = H[j]->s.d;
        hstate[j] = &H[j]->s;
    }

    double *d_jac = ensure_jac(dev, n_obs * n_tp);
    launch_fill_zero_doubles(dev, d_jac, n_obs * n_tp);
    std::vector<std::pair<size_t, double>> host_entries; // (flat index, value)

    const PlanPlace pl = place_in_arena(dev, img_r);
    ensure_parts(dev, parts.doubles);
    std::unique_ptr<TmpState> mu, lambda2;
    if (alt) {
        lambda2 = std::make_unique<TmpState>(n, ref.dtype, ref.device);
    }
    PhiPair phi{lambda.s, lambda2 ? lambda2->s : State{}};
    for (size_t i = 0; i < steps.size(); i++) {
        const Step &st = steps[i];
        if (enqueue_reverse_step(dev, phi, hptr.data(), n_obs, n_tp, st, img_r, i, pl, parts, d_jac)) {
            enqueue_flush(dev, parts, pl, i, n_obs, n_tp, d_jac);
            continue;
        }
        const PlanOp &p = st.single;
        if (p.trainable) {
            if (!mu) {
                mu = std::make_unique<TmpState>(n, ref.dtype, ref.device);
            }
            launch_copy(dev, mu->s, phi.cur);
        }
        apply_single(dev, phi.cur, p.U);
        if (p.trainable) {
            apply_generator_dev(dev, mu->s, p.G);
            std::vector<double> ri(2 * n_obs);
            inner_products(dev, hstate.data(), static_cast<int>(n_obs), mu->s, ri.data());
            for (size_t j = 0; j < n_obs; j++) {
                host_entries.push_back({j * n_tp + static_cast<size_t>(p.col),
                                        p.coef * ri[2 * j + 1]});
            }
        }
        for (size_t j = 0; j < n_obs; j++) {
            apply_single(dev, H[j]->s, p.U);
        }
        enqueue_flush(dev, parts, pl, i, n_obs, n_tp, d_jac);
    }
    PLK_HIP(hipMemcpyAsync(jac, d_jac, sizeof(double) * n_obs * n_tp, hipMemcpyDeviceToHost,
                           dev.stream));
    // Also keeps the host images alive until their copies have run.
    PLK_HIP(hipStreamSynchronize(dev.stream));
    for (auto &e : host_entries) {
        jac[e.first] = e.second;
    }
}

// ---------------------------------------------------------------------------
// Batched circuits: independent circuits, each from |0...0> with one
// observable, planned on the host into register-tile passes
// (kernels_batch.hip).
// ---------------------------------------------------------------------------
struct BatchInput {
    int n = 0;
    const OpsData *ops = nullptr;
    const ObsNode *obs = nullptr;
    std::vector<size_t> tp;
};

// A planned batch circuit: ranges in its part's tables.
struct BatchPlanned {
    int n = 0;
    std::pair<int, int> fwd, rev;
    int term_first = 0, term_count = 0;
    int64_t jac = 0;  // first Jacobian entry
    double cost = 0.0;
    bool staged = false;
};

// The circuits one host thread planned.
struct BatchPart {
    SweepTables t;
    std::vector<BatchPlanned> circuits;
    int64_t nparams = 0;
    int64_t jac_len = 0;
};

// Widest circuit that runs whole in one workgroup: eight tiles, one per wave.
// Wider ones run pass by pass over many workgroups (a 16-qubit, 8-layer
// circuit takes 32 ms in one workgroup of LDS tiles).
int batch_whole_qubits(int dtype) {
    return env_int("PLK_BATCH_WHOLE_QUBITS", sweep_reg_bits(dtype) + RT_LANE_BITS + 3);
}

void plan_batch_circuit(BatchPart &bp, const BatchInput &in, int dtype) {
    const int n = in.n;
    const OpsData &ops = *in.ops;
    BatchPlanned c;
    c.n = n;
    c.jac = bp.jac_len;
    std::vector<PauliTerm> pt;
    if (!to_pauli(*in.obs, n, pt)) {
        raise(PLK_ERR_UNSUPPORTED,
              "batched circuits support observables that are sums of Pauli words");
    }
    c.term_first = static_cast<int>(bp.t.terms.size());
    c.term_count = static_cast<int>(pt.size());
    for (const auto &t : pt) {
        bp.t.terms.push_back({static_cast<uint32_t>(t.x), static_cast<uint32_t>(t.zy), t.coeff.real(),
                              t.coeff.imag()});
    }
    std::vector<int32_t> pidx(ops.names.size(), -1);
    int64_t np = bp.nparams;
    for (size_t i = 0; i < ops.names.size(); i++) {
        if (!ops.params[i].empty()) {
            pidx[i] = static_cast<int32_t>(np++);
        }
    }
    if (np > INT32_MAX) {
        raise(PLK_ERR_UNSUPPORTED, "batched parameters exceed 2^31");
    }
    bp.nparams = np;
    auto mark = [&](PlanOp &p, size_t i, bool adj) {
        if (p.U.wires.size() != 1) {
            return;
        }
        RunGate g;
        const int16_t kind = patch_gate_of(ops, i);
        g.g.gate = kind == BPG_NONE ? static_cast<int16_t>(BPG_CONST) : kind;
        g.g.adj = adj ? 1 : 0;
        g.g.param = pidx[i];
        g.g.coef = p.trainable ? p.coef : 0.0;
        if (kind == BPG_NONE) {
            prepare(p);
            g.mat = p.U.mat;
        }
        p.gates = {std::move(g)};
    };
    std::vector<PlanOp> rev = reverse_ops(ops, in.tp, n, dtype);
    for (auto &p : rev) {
        mark(p, static_cast<size_t>(p.src), p.adj);
    }
    std::vector<PlanOp> fwd = forward_ops(ops, n);
    for (size_t i = 0; i < fwd.size(); i++) {
        mark(fwd[i], i, ops.inverses[i]);
    }
    const int L = n > batch_whole_qubits(dtype) ? low_bits(dtype) : 0;
    c.fwd = bp.t.add(std::move(fwd), n, dtype, L, true);
    c.rev = bp.t.add(std::move(rev), n, dtype, L, true);
    c.staged = L > 0 && c.fwd.second > 0 && n > sweep_reg_bits(dtype) + RT_LANE_BITS;
    for (int p = c.fwd.first; p < c.rev.first + c.rev.second; p++) {
        c.cost += bp.t.passes[p].ninstr * (p < c.rev.first ? 1.0 : 2.0) * std::ldexp(1.0, std::max(0, n - 8));
    }
    bp.jac_len += static_cast<int64_t>(in.tp.size());
    bp.circuits.push_back(c);
}

// Where a part's tables begin among the batch's.
struct BatchBase {
    int32_t pass = 0, entry = 0, term = 0, run = 0, gate = 0, mat = 0, param = 0;
    int64_t prog = 0, jac = 0;
};

BatchBase after(const BatchBase &b, const BatchPart &p) {
    auto sum = [](int32_t x, int64_t y) {
        if (x + y > INT32_MAX) {
            raise(PLK_ERR_UNSUPPORTED, "batch tables exceed 2^31 rows");
        }
        return static_cast<int32_t>(x + y);
    };
    BatchBase n;
    n.pass = sum(b.pass, static_cast<int64_t>(p.t.passes.size()));
    n.entry = sum(b.entry, static_cast<int64_t>(p.t.entries.size()));
    n.term = sum(b.term, static_cast<int64_t>(p.t.terms.size()));
    n.run = sum(b.run, static_cast<int64_t>(p.t.runs.size()));
    n.gate = sum(b.gate, static_cast<int64_t>(p.t.gates.size()));
    n.mat = sum(b.mat, static_cast<int64_t>(p.t.consts.size() / 8));
    n.param = sum(b.param, p.nparams);
    n.prog = (b.prog + static_cast<int64_t>(p.t.blob.size()) + 255) & ~int64_t{255};
    n.jac = b.jac + p.jac_len;
    return n;
}

// The batch's tables in one image, each part's written where it belongs with
// its indices rebased.
struct BatchImage {
    size_t passes, entries, terms, runs, gates, consts, prog; // bytes from the image's start

    void put(unsigned char *img, const BatchPart &part, const BatchBase &b) const {
        const SweepTables &t = part.t;
        auto *P = reinterpret_cast<SweepPass *>(img + passes) + b.pass;
        for (SweepPass p : t.passes) {
            p.prog += b.prog;
            p.entry_first += b.entry;
            *P++ = p;
        }
        auto *R = reinterpret_cast<BatchRun *>(img + runs) + b.run;
        for (BatchRun r : t.runs) {
            r.ins += b.prog;
            r.first += b.gate;
            r.entry += r.entry < 0 ? 0 : b.entry;
            *R++ = r;
        }
        auto *G = reinterpret_cast<BatchGate *>(img + gates) + b.gate;
        for (BatchGate g : t.gates) {
            g.param += g.gate == BPG_CONST ? b.mat : b.param;
            *G++ = g;
        }
        auto copy = [&](size_t at, const void *src, size_t bytes) {
            if (bytes > 0) {
                std::memcpy(img + at, src, bytes);
            }
        };
        copy(entries + static_cast<size_t>(b.entry) * sizeof(SweepEntry), t.entries.data(),
             t.entries.size() * sizeof(SweepEntry));
        copy(terms + static_cast<size_t>(b.term) * sizeof(SweepTerm), t.terms.data(),
             t.terms.size() * sizeof(SweepTerm));
        copy(consts + static_cast<size_t>(b.mat) * 8 * sizeof(double), t.consts.data(),
             t.consts.size() * sizeof(double));
        copy(prog + static_cast<size_t>(b.prog), t.blob.data(), t.blob.size());
    }
};

// Runs fn(t, lo, hi) for nthreads contiguous ranges of [0, count) on host
// threads (inline when there is one).
template <typename F> void parallel_ranges(size_t count, size_t nthreads, F fn) {
    nthreads = std::max<size_t>(1, std::min(nthreads, count));
    if (nthreads == 1) {
        fn(size_t{0}, size_t{0}, count);
        return;
    }
    std::vector<std::thread> pool;
    for (size_t t = 0; t < nthreads; t++) {
        pool.emplace_back(fn, t, count * t / nthreads, count * (t + 1) / nthreads);
    }
    for (auto &th : pool) {
        th.join();
    }
}

size_t plan_threads(size_t count) {
    const size_t hw = std::max(1u, std::thread::hardware_concurrency());
    return std::min<size_t>(
        {static_cast<size_t>(std::max(1, env_int("PLK_PLAN_THREADS", static_cast<int>(hw)))),
         (count + 31) / 32, size_t{64}});
}

// Everything a batch plan depends on except the angles of patched gates:
// qubits, op names / wires / inverse flags, the values of every other
// parameter and matrix, the trainable set and the observable.
uint64_t circuit_key(const BatchInput &in) {
    Hasher H;
    H.add(static_cast<uint64_t>(in.n));
    H.add(ops_key(*in.ops));
    H.add(static_cast<uint64_t>(in.tp.size()));
    for (auto t : in.tp) {
        H.add(static_cast<uint64_t>(t));
    }
    H.add(obs_key(*in.obs));
    return H.h;
}

// Circuits whose states fit the scratch together, run by one sequence of
// launches: the whole circuits' jobs, then the staged ones' launches.
struct BatchGroup {
    struct Launch {
        BatchStage stage;
        size_t first;
        int count; // blocks
    };
    struct Jobs {
        size_t first;
        int count, waves;
    };
    std::vector<Jobs> whole;
    std::vector<Launch> staged;
    size_t tail_first = 0;
    int tail_count = 0;
};

// The last batch plan of one precision, resident on its device: tables,
// patch list, parameter slots, scratch and result buffers in one allocation.
// A call whose circuits have the same keys reuses it and uploads only the
// parameters; any other call replaces it.
struct BatchCache {
    bool valid = false;
    int device = -1;
    int whole_qubits = 0;
    std::vector<uint64_t> keys;
    std::vector<int64_t> param_base; // first global parameter of each circuit
    std::vector<BatchGroup> groups;
    int64_t nparams = 0, nruns = 0;
    int64_t jac_len = 0;
    void *dbuf = nullptr;
    unsigned char *blob = nullptr;
    SweepEntry *entries = nullptr;
    const BatchRun *runs = nullptr;
    const BatchGate *gates = nullptr;
    const double *consts = nullptr;
    double *params = nullptr;
    const SweepJob *jobs = nullptr;
    const BatchBlock *blocks = nullptr;
    const BatchTail *tails = nullptr;
    BatchArgs A{};

    void release() {
        valid = false;
        if (dbuf != nullptr) {
            PLK_HIP(hipStreamSynchronize(device_stream()));
            PLK_HIP(hipFree(dbuf));
            dbuf = nullptr;
        }
    }
    hipStream_t device_stream() const { return ::plk::device(device).stream; }
};

BatchCache &batch_cache(int dtype) {
    static BatchCache c64, c128; // released with the process
    return dtype == PLK_C64 ? c64 : c128;
}

// Amplitudes of scratch (phi and h of every circuit of a group).
constexpr int64_t kBatchScratch = int64_t{1} << 29;
// Blocks of a staged circuit's launches: a wave per tile up to 64.
constexpr int kBatchBlocks = 64;

// Plans every circuit and makes the result resident in C.
// Every validation error is raised while planning, before any device call.
void build_batch_cache(BatchCache &C, int dtype, int device_id, const std::vector<BatchInput> &in) {
    const size_t nthreads = plan_threads(in.size());
    std::unique_ptr<HostScope> phase = std::make_unique<HostScope>("host_batch_plan");
    std::vector<BatchPart> parts(nthreads);
    std::vector<std::pair<size_t, Error>> failures(nthreads, {SIZE_MAX, Error{PLK_OK, ""}});
    parallel_ranges(in.size(), nthreads, [&](size_t t, size_t lo, size_t hi) {
        for (size_t i = lo; i < hi; i++) {
            try {
                plan_batch_circuit(parts[t], in[i], dtype);
            } catch (const Error &e) {
                failures[t] = {i, e};
                return;
            } catch (const std::exception &e) {
                failures[t] = {i, Error{PLK_ERR_INVALID, e.what()}};
                return;
            }
        }
    });
    for (const auto &f : failures) {
        if (f.first != SIZE_MAX) {
            raise(f.second.code, "circuit " + std::to_string(f.first) + ": " + f.second.msg);
        }
    }
    phase = std::make_unique<HostScope>("host_batch_pack");
    std::vector<BatchBase> base(parts.size() + 1);
    std::vector<BatchPlanned> circuits; // ranges within their part's tables
    std::vector<int32_t> part_of;
    circuits.reserve(in.size());
    for (size_t t = 0; t < parts.size(); t++) {
        base[t + 1] = after(base[t], parts[t]);
        for (const BatchPlanned &c : parts[t].circuits) {
            circuits.push_back(c);
            circuits.back().jac += base[t].jac;
            part_of.push_back(static_cast<int32_t>(t));
        }
    }
    const BatchBase &all = base.back();
    auto passes = [&](int32_t ci, const std::pair<int, int> &r) { // in the batch's table
        return std::pair<int, int>{r.first + base[part_of[ci]].pass, r.second};
    };
    Device &dev = device(device_id);
    C.release();
    C.device = dev.id;
    C.groups.clear();

    // Costliest circuits first, so that a launch ends together.
    std::vector<int32_t> by_cost(in.size());
    for (size_t i = 0; i < in.size(); i++) {
        by_cost[i] = static_cast<int32_t>(i);
    }
    std::stable_sort(by_cost.begin(), by_cost.end(),
                     [&](int32_t a, int32_t b) { return circuits[a].cost > circuits[b].cost; });
    std::vector<SweepJob> jobs;         // pointers are set once the buffer exists
    std::vector<int32_t> job_circuit;
    std::vector<std::pair<int64_t, int64_t>> job_state; // phi, h amplitudes
    std::vector<BatchCircuit> staged;
    std::vector<BatchBlock> blocks;
    std::vector<BatchTail> tails;
    const int tile = sweep_reg_bits(dtype) + RT_LANE_BITS;
    {
        size_t nblocks = 0, ntails = 0;
        for (size_t i = 0; i < circuits.size(); i++) {
            const BatchPlanned &c = circuits[i];
            if (!c.staged) {
                continue;
            }
            nblocks += static_cast<size_t>(c.fwd.second + c.rev.second + 1) *
                       static_cast<size_t>(std::min(kBatchBlocks, 1 << (c.n - tile)));
            ntails += 1 + in[i].tp.size();
        }
        blocks.reserve(nblocks);
        tails.reserve(ntails);
    }
    int64_t amps_max = 0, parts_max = 0;
    for (size_t at = 0; at < by_cost.size();) {
        BatchGroup g;
        int64_t amps = 0, psum = 0;
        std::vector<int32_t> members;
        while (at < by_cost.size()) {
            const int64_t need = int64_t{2} << circuits[by_cost[at]].n;
            if (!members.empty() && amps + need > kBatchScratch) {
                break;
            }
            members.push_back(by_cost[at++]);
            amps += need;
        }
        amps_max = std::max(amps_max, amps);
        amps = 0;
        // Whole circuits, several tiles first; each launch has the waves of its widest.
        for (const bool wide : {true, false}) {
            BatchGroup::Jobs l{jobs.size(), 0, 1};
            for (int32_t ci : members) {
                const BatchPlanned &c = circuits[ci];
                if (c.staged || (c.n > tile) != wide) {
                    continue;
                }
                SweepJob J{};
                J.n = c.n;
                std::tie(J.fwd_first, J.fwd_count) = passes(ci, c.fwd);
                std::tie(J.rev_first, J.rev_count) = passes(ci, c.rev);
                J.term_first = c.term_first + base[part_of[ci]].term;
                J.term_count = c.term_count;
                J.jac_len = static_cast<int32_t>(in[ci].tp.size());
                jobs.push_back(J);
                job_circuit.push_back(ci);
                job_state.push_back({amps, amps + (int64_t{1} << c.n)});
                amps += int64_t{2} << c.n;
                l.count++;
                l.waves = std::max(l.waves, sweep_waves(c.n, dtype));
            }
            if (l.count > 0) {
                g.whole.push_back(l);
            }
        }
        // Staged circuits.
        std::vector<int32_t> ids; // positions in `staged`
        std::vector<int32_t> who;         // and the circuits there
        int nfwd = 0, nrev = 0;
        g.tail_first = tails.size();
        for (int32_t ci : members) {
            const BatchPlanned &c = circuits[ci];
            if (!c.staged) {
                continue;
            }
            BatchCircuit b{};
            b.phi = amps;
            b.h = amps + (int64_t{1} << c.n);
            amps += int64_t{2} << c.n;
            b.n = c.n;
            b.blocks = std::min(kBatchBlocks, 1 << (c.n - tile));
            b.term_first = c.term_first + base[part_of[ci]].term;
            b.term_count = c.term_count;
            b.eparts = psum;
            psum += b.blocks;
            tails.push_back({b.eparts, ci, -1, b.blocks});
            for (int p = c.rev.first; p < c.rev.first + c.rev.second; p++) {
                SweepPass &P = parts[part_of[ci]].t.passes[p];
                P.parts = psum;
                psum += static_cast<int64_t>(P.nslots) * b.blocks;
                for (int e = 0; e < P.entry_count; e++) {
                    tails.push_back({P.parts, c.jac, base[part_of[ci]].entry + P.entry_first + e, b.blocks});
                }
            }
            nfwd = std::max(nfwd, c.fwd.second);
            nrev = std::max(nrev, c.rev.second);
            ids.push_back(static_cast<int32_t>(staged.size()));
            who.push_back(ci);
            staged.push_back(b);
        }
        auto launch = [&](BatchStage stage, int k) {
            BatchGroup::Launch l{stage, blocks.size(), 0};
            for (size_t q = 0; q < ids.size(); q++) {
                const BatchPlanned &c = circuits[who[q]];
                const std::pair<int, int> r = passes(who[q], stage == BATCH_FORWARD ? c.fwd : c.rev);
                if (stage != BATCH_OBSERVABLE && k >= r.second) {
                    continue;
                }
                for (int x = 0; x < staged[ids[q]].blocks; x++) {
                    blocks.push_back({ids[q], stage == BATCH_OBSERVABLE ? 0 : r.first + k, x,
                                      stage == BATCH_FORWARD && k == 0 ? 1 : 0});
                }
            }
            l.count = static_cast<int>(blocks.size() - l.first);
            g.staged.push_back(l);
        };
        if (!ids.empty()) {
            for (int k = 0; k < nfwd; k++) {
                launch(BATCH_FORWARD, k);
            }
            launch(BATCH_OBSERVABLE, 0);
            for (int k = 0; k < nrev; k++) {
                launch(BATCH_REVERSE, k);
            }
        }
        g.tail_count = static_cast<int>(tails.size() - g.tail_first);
        parts_max = std::max(parts_max, psum);
        C.groups.push_back(std::move(g));
    }

    // The image: the parts' tables, written side by side by several threads, and
    // the schedule. Not a vector, whose zeroes would be written first.
    size_t bytes = 0;
    auto table = [&](size_t count, size_t size) {
        const size_t at = bytes;
        bytes = (bytes + count * size + 255) & ~size_t{255};
        return at;
    };
    BatchImage img;
    const size_t o_jobs = table(jobs.size(), sizeof(SweepJob));
    img.passes = table(static_cast<size_t>(all.pass), sizeof(SweepPass));
    img.entries = table(static_cast<size_t>(all.entry), sizeof(SweepEntry));
    img.terms = table(static_cast<size_t>(all.term), sizeof(SweepTerm));
    img.runs = table(static_cast<size_t>(all.run), sizeof(BatchRun));
    img.gates = table(static_cast<size_t>(all.gate), sizeof(BatchGate));
    img.consts = table(static_cast<size_t>(all.mat) * 8, sizeof(double));
    const size_t o_staged = table(staged.size(), sizeof(BatchCircuit));
    const size_t o_blocks = table(blocks.size(), sizeof(BatchBlock));
    const size_t o_tails = table(tails.size(), sizeof(BatchTail));
    img.prog = table(static_cast<size_t>(all.prog), 1);
    std::unique_ptr<unsigned char[]> host(new unsigned char[bytes]);
    parallel_ranges(parts.size(), parts.size(), [&](size_t, size_t lo, size_t hi) {
        for (size_t t = lo; t < hi; t++) {
            img.put(host.get(), parts[t], base[t]);
            parts[t] = BatchPart{};
        }
    });
    auto put = [&](size_t at, const auto &v) {
        if (!v.empty()) {
            std::memcpy(host.get() + at, v.data(), v.size() * sizeof(v[0]));
        }
    };
    put(o_staged, staged);
    put(o_blocks, blocks);
    put(o_tails, tails);
    auto up = [](size_t x) { return (x + 255) & ~size_t{255}; };
    const size_t amp = dtype == PLK_C64 ? 8 : 16;
    const size_t o_params = bytes;
    const size_t o_scratch = o_params + up(static_cast<size_t>(all.param) * sizeof(double));
    const size_t o_parts = o_scratch + up(static_cast<size_t>(amps_max) * amp);
    const size_t o_exp = o_parts + up(static_cast<size_t>(parts_max) * sizeof(double));
    const size_t o_jac = o_exp + up(in.size() * sizeof(double));
    const size_t total = o_jac + static_cast<size_t>(all.jac) * sizeof(double) + 256;

    phase = std::make_unique<HostScope>("host_batch_upload");
    C.dbuf = dev_malloc(dev.id, total, "batch plan");
    auto *w = static_cast<unsigned char *>(C.dbuf);
    auto *d_jac = reinterpret_cast<double *>(w + o_jac);
    auto *d_exp = reinterpret_cast<double *>(w + o_exp);
    for (size_t j = 0; j < jobs.size(); j++) {
        SweepJob &J = jobs[j];
        J.phi = w + o_scratch + static_cast<size_t>(job_state[j].first) * amp;
        J.h = w + o_scratch + static_cast<size_t>(job_state[j].second) * amp;
        J.jac = d_jac + circuits[job_circuit[j]].jac;
        J.expval = d_exp + job_circuit[j];
    }
    put(o_jobs, jobs);
    PLK_HIP(hipMemcpy(w, host.get(), bytes, hipMemcpyHostToDevice));
    record_kernel("host_batch_table_bytes", 0.f, static_cast<double>(bytes));

    BatchArgs &A = C.A;
    A.circuits = reinterpret_cast<const BatchCircuit *>(w + o_staged);
    A.passes = reinterpret_cast<const SweepPass *>(w + img.passes);
    A.entries = reinterpret_cast<const SweepEntry *>(w + img.entries);
    A.terms = reinterpret_cast<const SweepTerm *>(w + img.terms);
    A.blob = w + img.prog;
    A.scratch = w + o_scratch;
    A.parts = reinterpret_cast<double *>(w + o_parts);
    A.expvals = d_exp;
    A.jac = d_jac;
    C.blob = w + img.prog;
    C.entries = reinterpret_cast<SweepEntry *>(w + img.entries);
    C.runs = reinterpret_cast<const BatchRun *>(w + img.runs);
    C.nruns = all.run;
    C.gates = reinterpret_cast<const BatchGate *>(w + img.gates);
    C.consts = reinterpret_cast<const double *>(w + img.consts);
    C.params = reinterpret_cast<double *>(w + o_params);
    C.jobs = reinterpret_cast<const SweepJob *>(w + o_jobs);
    C.blocks = reinterpret_cast<const BatchBlock *>(w + o_blocks);
    C.tails = reinterpret_cast<const BatchTail *>(w + o_tails);
    C.nparams = all.param;
    C.jac_len = all.jac;
    C.param_base.assign(in.size(), 0);
    int64_t param = 0;
    for (size_t i = 0; i < in.size(); i++) {
        C.param_base[i] = param;
        param += static_cast<int64_t>(in[i].ops->num_par_ops());
    }
    C.valid = true;
}

void adjoint_batched_run(int dtype, int device_id, const std::vector<BatchInput> &in, double *expvals,
                         double *jac) {
    if (in.empty()) {
        return;
    }
    std::unique_ptr<HostScope> phase = std::make_unique<HostScope>("host_batch_key");
    // New matrices are hashed by several threads, each list's by one (circuits
    // may share it).
    std::vector<const OpsData *> fresh;
    for (const BatchInput &c : in) {
        if (c.ops->dense && !c.ops->keyed) {
            fresh.push_back(c.ops);
        }
    }
    std::sort(fresh.begin(), fresh.end(), std::less<const OpsData *>());
    fresh.erase(std::unique(fresh.begin(), fresh.end()), fresh.end());
    parallel_ranges(fresh.size(), plan_threads(fresh.size()), [&](size_t, size_t lo, size_t hi) {
        for (size_t i = lo; i < hi; i++) {
            ops_key(*fresh[i]);
        }
    });
    std::vector<uint64_t> keys(in.size());
    for (size_t i = 0; i < in.size(); i++) {
        keys[i] = circuit_key(in[i]);
    }
    phase.reset();
    BatchCache &C = batch_cache(dtype);
    const int whole = batch_whole_qubits(dtype);
    if (!(C.valid && C.device == device_id && C.whole_qubits == whole && C.keys == keys)) {
        C.valid = false;
        build_batch_cache(C, dtype, device_id, in);
        C.keys = std::move(keys);
        C.whole_qubits = whole;
    }
    Device &dev = device(device_id);

    // Angles of this call, in the plan's parameter order, then the patch
    // kernel rewrites every run with angles on the device.
    phase = std::make_unique<HostScope>("host_batch_params");
    std::vector<double> params(static_cast<size_t>(C.nparams));
    for (size_t c = 0; c < in.size(); c++) {
        const std::vector<double> &a = in[c].ops->angles;
        std::copy(a.begin(), a.end(), params.begin() + C.param_base[c]);
    }
    PLK_HIP(hipMemcpyAsync(C.params, params.data(), params.size() * sizeof(double),
                           hipMemcpyHostToDevice, dev.stream));
    phase = std::make_unique<HostScope>("host_batch_launch");
    launch_batch_patch(dev, dtype, C.blob, C.entries, C.runs, C.nruns, C.gates, C.params, C.consts);
    {
        ProfScope prof("adjoint_batch", 0.0, dev.stream);
        launch_fill_zero_doubles(dev, C.A.jac, static_cast<size_t>(C.jac_len));
        for (const BatchGroup &g : C.groups) {
            for (const auto &l : g.whole) {
                SweepArgs S;
                S.jobs = C.jobs + l.first;
                S.passes = C.A.passes;
                S.entries = C.A.entries;
                S.terms = C.A.terms;
                S.blob = C.A.blob;
                launch_sweep(dev, dtype, S, l.count, l.waves);
            }
            for (const auto &l : g.staged) {
                launch_batch_stage(dev, dtype, C.A, C.blocks + l.first, l.count, l.stage);
            }
            launch_batch_tails(dev, C.A, C.tails + g.tail_first, g.tail_count);
        }
    }
    phase = std::make_unique<HostScope>("host_batch_results");
    PLK_HIP(hipMemcpyAsync(expvals, C.A.expvals, in.size() * sizeof(double),
                           hipMemcpyDeviceToHost, dev.stream));
    if (C.jac_len > 0) {
        PLK_HIP(hipMemcpyAsync(jac, C.A.jac, static_cast<size_t>(C.jac_len) * sizeof(double),
                               hipMemcpyDeviceToHost, dev.stream));
    }
    // Also keeps `params` alive until its upload has been read.
    PLK_HIP(hipStreamSynchronize(dev.stream));
}

std::vector<size_t> to_vec(const size_t *w, size_t n) {
    return std::vector<size_t>(w, w + n);
}

std::vector<cd> to_cvec(const double *m, size_t len) {
    std::vector<cd> v(len);
    for (size_t i = 0; i < len; i++) {
        v[i] = cd{m[2 * i], m[2 * i + 1]};
    }
    return v;
}

State &S(plk_state *p) {
    if (!p) {
        raise(PLK_ERR_INVALID, "null state handle");
    }
    return p->s;
}

const State &S(const plk_state *p) {
    if (!p) {
        raise(PLK_ERR_INVALID, "null state handle");
    }
    return p->s;
}

} // namespace

} // namespace plk

struct plk_obs {
    std::shared_ptr<const plk::ObsNode> node;
};

struct plk_ops {
    plk::OpsData data;
};

using namespace plk;

#define PLK_TRY(body)                                                          \
    try {                                                                      \
        std::lock_guard<std::recursive_mutex> plk_engine_lock_(engine_mutex()); \
        begin_call();                                                          \
        body;                                                                  \
        g_last_error.clear();                                                  \
        return PLK_OK;                                                         \
    } catch (const plk::Error &e) {                                            \
        g_last_error = e.msg;                                                  \
        return e.code;                                                         \
    } catch (const std::bad_alloc &) {                                         \
        g_last_error = "host allocation failed";                               \
        return PLK_ERR_OOM;                                                    \
    } catch (const std::exception &e) {                                        \
        g_last_error = e.what();                                               \
        return PLK_ERR_INVALID;                                                \
    }

static const ObsNode &O(const plk_obs *o) {
    if (!o || !o->node) {
        raise(PLK_ERR_INVALID, "null observable handle");
    }
    return *o->node;
}

extern "C" {

const char *plk_last_error(void) { return g_last_error.c_str(); }

int plk_device_count(int *out) {
    PLK_TRY({
        int c = 0;
        PLK_HIP(hipGetDeviceCount(&c));
        *out = c;
    })
}

int plk_print_configuration(char *buf, size_t len) {
    PLK_TRY({
        std::ostringstream os;
        int count = 0;
        PLK_HIP(hipGetDeviceCount(&count));
        os << "plk_amd state-vector engine\n";
        os << "  HIP runtime devices: " << count << "\n";
        for (int d = 0; d < count; d++) {
            hipDeviceProp_t p;
            PLK_HIP(hipGetDeviceProperties(&p, d));
            os << "  device " << d << ": " << p.name << " arch=" << p.gcnArchName
               << " CUs=" << p.multiProcessorCount
               << " HBM=" << (p.totalGlobalMem >> 20) << " MiB"
               << " LDS/block=" << p.sharedMemPerBlock << " B"
               << " wavefront=" << p.warpSize << "\n";
        }
        os << "  build: gfx950 HIP kernels, complex64/complex128 states, FP64 reductions\n";
        os << "  fused segments: up to " << SEG_KMAX << " wires, " << SEG_PMAX
           << " trainable ops and " << SEG_NJMAX << " observable states per HBM pass\n";
        const std::string s = os.str();
        if (len > 0) {
            std::strncpy(buf, s.c_str(), len - 1);
            buf[len - 1] = '\0';
        }
    })
}

int plk_state_create(int num_qubits, int dtype, int device_id, plk_state **out) {
    PLK_TRY({
        if (num_qubits < 0 || num_qubits > 40) {
            raise(PLK_ERR_INVALID, "number of qubits out of range");
        }
        if (dtype != PLK_C64 && dtype != PLK_C128) {
            raise(PLK_ERR_INVALID, "dtype must be PLK_C64 or PLK_C128");
        }
        Device &dev = device(device_id);
        auto h = std::make_unique<plk_state>();
        h->s.n = num_qubits;
        h->s.dtype = dtype;
        h->s.len = size_t{1} << num_qubits;
        h->s.device = device_id;
        h->s.d = dev_malloc(device_id, h->s.bytes(), "state vector");
        launch_set_basis(dev, h->s, 0);
        PLK_HIP(hipStreamSynchronize(dev.stream));
        *out = h.release();
    })
}

int plk_state_destroy(plk_state *sv) {
    PLK_TRY({
        if (sv) {
            Device &dev = device(sv->s.device);
            PLK_HIP(hipStreamSynchronize(dev.stream));
            PLK_HIP(hipFree(sv->s.d));
            delete sv;
        }
    })
}

int plk_state_num_qubits(const plk_state *sv, int *out) { PLK_TRY({ *out = S(sv).n; }) }

int plk_state_length(const plk_state *sv, size_t *out) { PLK_TRY({ *out = S(sv).len; }) }

int plk_state_dtype(const plk_state *sv, int *out) { PLK_TRY({ *out = S(sv).dtype; }) }

int plk_state_device_ptr(plk_state *sv, void **out) { PLK_TRY({ *out = S(sv).d; }) }

int plk_state_upload(plk_state *sv, const void *host, size_t length) {
    PLK_TRY({
        State &s = S(sv);
        if (length != s.len) {
            raise(PLK_ERR_INVALID, "HostToDevice: length " + std::to_string(length) +
                                       " does not match the state length " +
                                       std::to_string(s.len));
        }
        Device &dev = dev_of(s);
        PLK_HIP(hipMemcpyAsync(s.d, host, s.bytes(), hipMemcpyHostToDevice, dev.stream));
        PLK_HIP(hipStreamSynchronize(dev.stream));
    })
}

int plk_state_download(const plk_state *sv, void *host, size_t length) {
    PLK_TRY({
        const State &s = S(sv);
        if (length != s.len) {
            raise(PLK_ERR_INVALID, "DeviceToHost: length " + std::to_string(length) +
                                       " does not match the state length " +
                                       std::to_string(s.len));
        }
        Device &dev = dev_of(s);
        PLK_HIP(hipMemcpyAsync(host, s.d, s.bytes(), hipMemcpyDeviceToHost, dev.stream));
        PLK_HIP(hipStreamSynchronize(dev.stream));
    })
}

int plk_state_reset(plk_state *sv) {
    PLK_TRY({
        State &s = S(sv);
        launch_set_basis(dev_of(s), s, 0);
    })
}

int plk_state_set_basis(plk_state *sv, size_t index) {
    PLK_TRY({
        State &s = S(sv);
        if (index >= s.len) {
            raise(PLK_ERR_INVALID, "basis-state index out of range");
        }
        launch_set_basis(dev_of(s), s, index);
    })
}

int plk_state_set_values(plk_state *sv, const size_t *indices, const void *values,
                         size_t count) {
    PLK_TRY({
        State &s = S(sv);
        Device &dev = dev_of(s);
        for (size_t i = 0; i < count; i++) {
            if (indices[i] >= s.len) {
                raise(PLK_ERR_INVALID, "setStateVector: index out of range");
            }
        }
        launch_fill_zero(dev, s);
        if (count) {
            void *blob = nullptr;
            const size_t ib = count * sizeof(size_t);
            const size_t vo = (ib + 255) / 256 * 256;
            PLK_HIP(hipMalloc(&blob, vo + count * s.elem_bytes()));
            PLK_HIP(hipMemcpy(blob, indices, ib, hipMemcpyHostToDevice));
            PLK_HIP(hipMemcpy(static_cast<char *>(blob) + vo, values, count * s.elem_bytes(),
                              hipMemcpyHostToDevice));
            launch_scatter(dev, s, static_cast<const size_t *>(blob),
                           static_cast<char *>(blob) + vo, count);
            PLK_HIP(hipStreamSynchronize(dev.stream));
            PLK_HIP(hipFree(blob));
        }
    })
}

int plk_state_copy(plk_state *dst, const plk_state *src) {
    PLK_TRY({
        State &d = S(dst);
        const State &s = S(src);
        if (d.device != s.device) {
            raise(PLK_ERR_INVALID, "state copy across devices is not supported");
        }
        launch_copy(dev_of(d), d, s);
    })
}

int plk_state_synchronize(const plk_state *sv) {
    PLK_TRY({ PLK_HIP(hipStreamSynchronize(dev_of(S(sv)).stream)); })
}

int plk_apply(plk_state *sv, const char *name, const size_t *wires, size_t num_wires,
              int inverse, const double *params, size_t num_params) {
    PLK_TRY({
        State &s = S(sv);
        const std::string nm(name ? name : "");
        if (!is_named_gate(nm)) {
            raise(PLK_ERR_UNSUPPORTED, "operation " + nm + " has no named kernel");
        }
        std::vector<double> p(params, params + num_params);
        apply_single(dev_of(s), s,
                     compile_op(nm, to_vec(wires, num_wires), inverse != 0, p, {}, s.n));
    })
}

int plk_apply_matrix(plk_state *sv, const double *matrix, const size_t *wires,
                     size_t num_wires, int inverse) {
    PLK_TRY({
        State &s = S(sv);
        const size_t dim = size_t{1} << num_wires;
        apply_single(dev_of(s), s,
                     compile_op("Matrix", to_vec(wires, num_wires), inverse != 0, {},
                                to_cvec(matrix, dim * dim), s.n));
    })
}

int plk_apply_ops(plk_state *sv, const plk_ops *ops) {
    PLK_TRY({
        State &s = S(sv);
        if (!ops) {
            raise(PLK_ERR_INVALID, "null ops handle");
        }
        Device &dev = dev_of(s);
        std::vector<PlanOp> v = forward_ops(ops->data, s.n);
        if (sweep_serves(s) && sweep_pays_forward(s, v.size()) && sweep_takes(v)) {
            sweep_forward(dev, s, std::move(v));
        } else {
            run_forward(dev, s, forward_plan(dev, std::move(v), s.n, s.dtype, true));
        }
    })
}

int plk_apply_ops_blocks(plk_state *sv, const plk_ops *ops, size_t *num_blocks) {
    PLK_TRY({
        State &s = S(sv);
        if (!ops) {
            raise(PLK_ERR_INVALID, "null ops handle");
        }
        if (s.n < 9) {
            raise(PLK_ERR_UNSUPPORTED, "5-qubit MFMA blocks need at least 9 qubits");
        }
        const OpsData &d = ops->data;
        std::vector<CompiledOp> cops;
        cops.reserve(d.names.size());
        for (size_t i = 0; i < d.names.size(); i++) {
            cops.push_back(compile_op(d.names[i], d.wires[i], d.inverses[i], d.params[i],
                                      d.matrices[i], s.n));
        }
        const std::vector<FusedBlock> blocks = fuse_blocks(cops, s.n);
        apply_blocks(dev_of(s), s, blocks);
        if (num_blocks) {
            *num_blocks = blocks.size();
        }
    })
}

int plk_apply_generator(plk_state *sv, const char *name, const size_t *wires,
                        size_t num_wires, int adjoint, double *scale) {
    PLK_TRY({
        (void)adjoint;
        State &s = S(sv);
        CompiledGen g = compile_generator(name ? name : "", to_vec(wires, num_wires), s.n);
        apply_generator_dev(dev_of(s), s, g);
        *scale = g.scale;
    })
}

int plk_expval_named(const plk_state *sv, const char *name, const size_t *wires,
                     size_t num_wires, double *out) {
    PLK_TRY({
        const State &s = S(sv);
        ObsNode o;
        o.kind = ObsNode::Named;
        o.name = name ? name : "";
        o.wires = to_vec(wires, num_wires);
        std::vector<PauliTerm> terms;
        if (!to_pauli(o, s.n, terms)) {
            raise(PLK_ERR_INVALID, "named observable " + o.name + " is not supported");
        }
        *out = pauli_expval(dev_of(s), s, terms);
    })
}

int plk_expval_matrix(const plk_state *sv, const double *matrix, const size_t *wires,
                      size_t num_wires, double *out) {
    PLK_TRY({
        const State &s = S(sv);
        ObsNode o;
        o.kind = ObsNode::Hermitian;
        o.wires = to_vec(wires, num_wires);
        const size_t dim = size_t{1} << num_wires;
        o.matrix = to_cvec(matrix, dim * dim);
        *out = expval_obs(dev_of(s), s, o);
    })
}

int plk_expval_csr(const plk_state *sv, const double *data, const int64_t *indices,
                   const int64_t *indptr, size_t nnz, size_t num_rows, double *out) {
    PLK_TRY({
        const State &s = S(sv);
        CsrView v;
        v.data = data;
        v.indices = indices;
        v.indptr = indptr;
        v.idx32 = false;
        v.nnz = nnz;
        v.rows = num_rows;
        *out = csr_expval_once(dev_of(s), s, v);
    })
}

int plk_expval_csr_i32(const plk_state *sv, const double *data, const int32_t *indices,
                       const int32_t *indptr, size_t nnz, size_t num_rows, double *out) {
    PLK_TRY({
        const State &s = S(sv);
        if (num_rows > size_t{1} << 31 || nnz > static_cast<size_t>(INT32_MAX)) {
            raise(PLK_ERR_INVALID, "CSR matrix too large for 32-bit indices");
        }
        CsrView v;
        v.data = data;
        v.indices = indices;
        v.indptr = indptr;
        v.idx32 = true;
        v.nnz = nnz;
        v.rows = num_rows;
        *out = csr_expval_once(dev_of(s), s, v);
    })
}

int plk_expval_obs(const plk_state *sv, const plk_obs *ob, double *out) {
    PLK_TRY({
        const State &s = S(sv);
        *out = expval_obs(dev_of(s), s, O(ob));
    })
}

int plk_expval_obs_noalloc(const plk_state *sv, const plk_obs *ob, double *out) {
    PLK_TRY({
        const State &s = S(sv);
        std::vector<PauliTerm> terms;
        // Expanded past the limit so that an oversized sum is reported by size.
        if (!to_pauli(O(ob), s.n, terms, 4 * kNoAllocMaxPauliWords)) {
            raise(PLK_ERR_UNSUPPORTED,
                  "plk_expval_obs_noalloc: the observable is not a sum of at most " +
                      std::to_string(kNoAllocMaxPauliWords) +
                      " products of Identity / PauliX / PauliY / PauliZ / Hadamard");
        }
        *out = pauli_expval_noalloc(dev_of(s), s, terms);
    })
}

int plk_inner_product(const plk_state *x, const plk_state *y, double *re, double *im) {
    PLK_TRY({
        const State &a = S(x);
        const State &b = S(y);
        if (a.len != b.len || a.dtype != b.dtype) {
            raise(PLK_ERR_INVALID, "inner product of states with different shapes");
        }
        const State *xs[1] = {&a};
        double ri[2];
        inner_products(dev_of(b), xs, 1, b, ri);
        *re = ri[0];
        *im = ri[1];
    })
}

int plk_obs_named(const char *name, const size_t *wires, size_t num_wires, plk_obs **out) {
    PLK_TRY({
        auto n = std::make_shared<ObsNode>();
        n->kind = ObsNode::Named;
        n->name = name ? name : "";
        n->wires = to_vec(wires, num_wires);
        note_obs(*n);
        *out = new plk_obs{n};
    })
}

int plk_obs_hermitian(const double *matrix, const size_t *wires, size_t num_wires,
                      plk_obs **out) {
    PLK_TRY({
        auto n = std::make_shared<ObsNode>();
        n->kind = ObsNode::Hermitian;
        n->wires = to_vec(wires, num_wires);
        const size_t dim = size_t{1} << num_wires;
        n->matrix = to_cvec(matrix, dim * dim);
        note_obs(*n);
        *out = new plk_obs{n};
    })
}

int plk_obs_tensor(const plk_obs *const *factors, size_t num_factors, plk_obs **out) {
    PLK_TRY({
        auto n = std::make_shared<ObsNode>();
        n->kind = ObsNode::Tensor;
        std::set<size_t> seen;
        for (size_t i = 0; i < num_factors; i++) {
            const ObsNode &f = O(factors[i]);
            for (auto w : obs_wires(f)) {
                if (!seen.insert(w).second) {
                    raise(PLK_ERR_INVALID, "All wires in observables must be disjoint.");
                }
            }
            n->terms.push_back(factors[i]->node);
        }
        note_obs(*n);
        *out = new plk_obs{n};
    })
}

int plk_obs_hamiltonian(const double *coeffs, const plk_obs *const *terms, size_t num_terms,
                        plk_obs **out) {
    PLK_TRY({
        auto n = std::make_shared<ObsNode>();
        n->kind = ObsNode::Hamiltonian;
        for (size_t i = 0; i < num_terms; i++) {
            O(terms[i]);
            n->terms.push_back(terms[i]->node);
            n->coeffs.push_back(coeffs[i]);
        }
        note_obs(*n);
        *out = new plk_obs{n};
    })
}

int plk_obs_sparse(const double *data, const int64_t *indices, const int64_t *indptr,
                   size_t nnz, size_t num_rows, const size_t *wires, size_t num_wires,
                   plk_obs **out) {
    PLK_TRY({
        auto n = std::make_shared<ObsNode>();
        n->kind = ObsNode::Sparse;
        n->data.assign(data, data + 2 * nnz);
        n->indices.assign(indices, indices + nnz);
        n->indptr.assign(indptr, indptr + num_rows + 1);
        n->rows = num_rows;
        n->wires = to_vec(wires, num_wires);
        note_obs(*n);
        *out = new plk_obs{n};
    })
}

int plk_obs_sparse_i32(const double *data, const int32_t *indices, const int32_t *indptr,
                       size_t nnz, size_t num_rows, const size_t *wires, size_t num_wires,
                       plk_obs **out) {
    PLK_TRY({
        if (num_rows > size_t{1} << 31 || nnz > static_cast<size_t>(INT32_MAX)) {
            raise(PLK_ERR_INVALID, "CSR matrix too large for 32-bit indices");
        }
        auto n = std::make_shared<ObsNode>();
        n->kind = ObsNode::Sparse;
        n->idx32 = true;
        n->data.assign(data, data + 2 * nnz);
        n->indices32.assign(indices, indices + nnz);
        n->indptr32.assign(indptr, indptr + num_rows + 1);
        n->rows = num_rows;
        n->wires = to_vec(wires, num_wires);
        note_obs(*n);
        *out = new plk_obs{n};
    })
}

int plk_obs_destroy(plk_obs *ob) { PLK_TRY({ delete ob; }) }

int plk_obs_wires(const plk_obs *ob, size_t *wires, size_t cap, size_t *count) {
    PLK_TRY({
        auto w = obs_wires(O(ob));
        *count = w.size();
        for (size_t i = 0; i < w.size() && i < cap; i++) {
            wires[i] = w[i];
        }
    })
}

int plk_obs_apply(plk_state *sv, const plk_obs *ob) {
    PLK_TRY({
        State &s = S(sv);
        Device &dev = dev_of(s);
        if (const PauliDevice *t = O(ob).pauli_on(dev, s.n)) {
            TmpState tmp(s.n, s.dtype, s.device);
            launch_pauli_apply(dev, tmp.s, s, *t);
            launch_copy(dev, s, tmp.s);
            PLK_HIP(hipStreamSynchronize(dev.stream));
        } else {
            apply_obs_general(dev, s, O(ob));
        }
    })
}

int plk_ops_create(size_t num_ops, const char *const *names, const double *params,
                   const size_t *param_offsets, const size_t *wires,
                   const size_t *wire_offsets, const int *inverses, const double *matrices,
                   const size_t *matrix_offsets, plk_ops **out) {
    PLK_TRY({
        auto h = std::make_unique<plk_ops>();
        OpsData &d = h->data;
        Hasher H;
        for (size_t i = 0; i < num_ops; i++) {
            d.names.emplace_back(names[i]);
            d.params.emplace_back(params + param_offsets[i], params + param_offsets[i + 1]);
            d.wires.emplace_back(wires + wire_offsets[i], wires + wire_offsets[i + 1]);
            d.inverses.push_back(inverses[i] != 0);
            const size_t ml = matrix_offsets[i + 1] - matrix_offsets[i];
            d.matrices.push_back(ml ? to_cvec(matrices + 2 * matrix_offsets[i], ml)
                                    : std::vector<cd>{});
            note_op(d, H, i);
        }
        *out = h.release();
    })
}

int plk_ops_destroy(plk_ops *ops) { PLK_TRY({ delete ops; }) }

int plk_ops_num_par_ops(const plk_ops *ops, size_t *out) {
    PLK_TRY({
        if (!ops) {
            raise(PLK_ERR_INVALID, "null ops handle");
        }
        *out = ops->data.num_par_ops();
    })
}

int plk_adjoint_jacobian(const plk_state *sv, const plk_obs *const *obs, size_t num_obs,
                         const plk_ops *ops, const size_t *trainable, size_t num_trainable,
                         int apply_operations, double *jac) {
    PLK_TRY({
        const State &s = S(sv);
        if (!ops) {
            raise(PLK_ERR_INVALID, "null ops handle");
        }
        std::vector<std::shared_ptr<const ObsNode>> ob;
        for (size_t j = 0; j < num_obs; j++) {
            O(obs[j]);
            ob.push_back(obs[j]->node);
        }
        std::vector<size_t> tp(trainable, trainable + num_trainable);
        adjoint_jacobian(s, ob, ops->data, tp, apply_operations != 0, jac);
    })
}

int plk_adjoint_batched(int dtype, int device_id, size_t num_circuits, const int *num_qubits,
                        const plk_ops *const *ops, const plk_obs *const *obs,
                        const size_t *const *trainable, const size_t *num_trainable,
                        double *expvals, double *jac) {
    PLK_TRY({
        if (dtype != PLK_C64 && dtype != PLK_C128) {
            raise(PLK_ERR_INVALID, "dtype must be PLK_C64 or PLK_C128");
        }
        if (num_circuits > 0 && (!num_qubits || !ops || !obs || !expvals)) {
            raise(PLK_ERR_INVALID, "null argument");
        }
        if (trainable && !num_trainable) {
            raise(PLK_ERR_INVALID, "trainable lists need their lengths");
        }
        HostScope whole("host_batch_call");
        std::vector<BatchInput> in(num_circuits);
        std::unique_ptr<HostScope> inputs = std::make_unique<HostScope>("host_batch_inputs");
        for (size_t i = 0; i < num_circuits; i++) {
            auto who = [i]() { return "circuit " + std::to_string(i) + ": "; };
            if (num_qubits[i] < 1 || num_qubits[i] > BATCH_NMAX) {
                raise(PLK_ERR_UNSUPPORTED, who() + "batched circuits have 1.." +
                                               std::to_string(BATCH_NMAX) + " qubits");
            }
            if (!ops[i]) {
                raise(PLK_ERR_INVALID, who() + "null ops handle");
            }
            in[i].n = num_qubits[i];
            in[i].ops = &ops[i]->data;
            in[i].obs = &O(obs[i]);
            if (trainable) {
                if (num_trainable[i] > 0 && !trainable[i]) {
                    raise(PLK_ERR_INVALID, who() + "null trainable list");
                }
                in[i].tp.assign(trainable[i], trainable[i] + num_trainable[i]);
            } else {
                in[i].tp.resize(ops[i]->data.num_par_ops());
                for (size_t k = 0; k < in[i].tp.size(); k++) {
                    in[i].tp[k] = k;
                }
            }
            if (in[i].tp.empty()) {
                raise(PLK_ERR_INVALID, who() + "No trainable parameters provided.");
            }
        }
        inputs.reset();
        if (num_circuits > 0 && !jac) {
            raise(PLK_ERR_INVALID, "null jac buffer");
        }
        adjoint_batched_run(dtype, device_id, in, expvals, jac);
    })
}

int plk_probs(const plk_state *sv, const size_t *wires, size_t num_wires, double *out) {
    PLK_TRY({
        const State &s = S(sv);
        if (!out || (num_wires > 0 && !wires)) {
            raise(PLK_ERR_INVALID, "null argument");
        }
        std::vector<size_t> w(wires, wires + num_wires);
        if (w.empty()) {
            for (int q = 0; q < s.n; q++) {
                w.push_back(static_cast<size_t>(q));
            }
        }
        uint64_t seen = 0;
        for (size_t q : w) {
            if (q >= static_cast<size_t>(s.n)) {
                raise(PLK_ERR_INVALID, "wire " + std::to_string(q) + " out of range");
            }
            if (seen >> q & 1) {
                raise(PLK_ERR_INVALID, "repeated wire in probs");
            }
            seen |= uint64_t{1} << q;
        }
        // The reference sums over the sorted wires and then transposes with
        // getTransposedIndexFunctor (MeasuresKokkos.hpp:487-512,
        // MeasuresFunctors.hpp:144-175); its output equals the marginal whose
        // index bits follow the wire order w[pi[pi[k]]], pi = argsort(w).
        std::vector<size_t> pi(w.size());
        for (size_t k = 0; k < pi.size(); k++) {
            pi[k] = k;
        }
        std::sort(pi.begin(), pi.end(), [&](size_t a, size_t b) { return w[a] < w[b]; });
        std::vector<int> g;
        for (size_t k = 0; k < w.size(); k++) {
            g.push_back(s.n - 1 - static_cast<int>(w[pi[pi[k]]]));
        }
        Device &dev = dev_of(s);
        set_device(s.device);
        probs(dev, s, g, out);
    })
}

int plk_generate_samples(const plk_state *sv, size_t num_shots, uint64_t seed, size_t *samples) {
    PLK_TRY({
        const State &s = S(sv);
        if (num_shots > 0 && !samples) {
            raise(PLK_ERR_INVALID, "null samples buffer");
        }
        Device &dev = dev_of(s);
        set_device(s.device);
        sample(dev, s, num_shots, seed, samples);
    })
}

int plk_profiling_enable(int on) { PLK_TRY({ profiling_enable_impl(on != 0); }) }

int plk_profiling_get(const char *kernel, double *launches, double *total_ms,
                      double *bytes) {
    PLK_TRY({
        KernelStats k = profiling_get_impl(kernel ? kernel : "");
        *launches = k.launches;
        *total_ms = k.ms;
        *bytes = k.bytes;
    })
}

int plk_profiling_names(char *buf, size_t len) {
    PLK_TRY({
        const std::string s = profiling_names_impl();
        if (len > 0) {
            std::strncpy(buf, s.c_str(), len - 1);
            buf[len - 1] = '\0';
        }
    })
}

} // extern "C"
