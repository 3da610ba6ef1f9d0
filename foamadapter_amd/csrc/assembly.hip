// assembly.hip -- the terms of one equation assembled in one pass
// (fv_assemble_terms): Euler ddt, div, laplacian, source, and an explicit
// divergence, into the matrix and one or three right-hand sides.
//
// Term by term, every assembly call reads and writes the whole matrix (values
// += on every entry) after four fills that clear it, computes each face's
// coefficient twice (once for either cell) from face arrays read by index, and a
// Vec3 equation assembles its one matrix three times.  What bounds the assembly is
// those bytes.  Here a workgroup of 256 cells computes each of its faces once, as
// the staged gathers of faceops.hip do (same lists, same LDS layout): the faces
// its cells own are streamed with coalesced loads, the lower faces owned by earlier
// workgroups come from the lists, and then each cell walks its faces in ascending
// order and writes its row, its diagonal and its right-hand sides once.  The row
// [lower | diagonal | upper] is the order of the walk, so no slot index is read.
//
// The sums of every term run over the cell's faces in the order of the single-term
// kernels of implicit.hip and the terms are added in the equation's order, so the
// values are the same bits.  150x140x130 cells: the momentum matrix with its three
// right-hand sides 2.1 ms term by term -> 151 us (718 MB at least: 4.8 TB/s), the
// pressure equation with its explicit divergence 390 -> 107 us (520 MB); 194 and 150
// before the rows went through LDS and the bricks were dealt to the XCDs in runs.
// Workgroups whose faces do not fit the LDS lists take
// the same walk with the coefficients recomputed per cell.
#include <type_traits>

#include "implicit.hpp"

using namespace fvhip;

namespace {

// Equation: which terms there are and their inputs.  coefficients: c*.
struct Terms {
    // cell terms
    const double* Told;   // ddt: interleaved [N, NC]
    double rdt, cDdt;
    const double* source; // [N]
    double cSource;
    // div
    const double* phi;
    int scheme;
    double cDiv;
    // laplacian
    const double* gamma;
    double cLap;
    // explicit div (surfaceIntegrate) of a flux
    const double* ephi;
    double cEdiv;
    // boundary values and gradients [B, NC] of the div and laplacian terms
    const int8_t* kind;
    const double *Tb, *Tg;
};

struct MeshIn {
    int N, F, nBlocks, run;
    const int32_t *nbr, *ownStart, *lowOff, *lowFace, *bOff, *bFace, *rowOffs;
    const double *V, *w, *magSf, *nodc, *magSfb, *dcb;
    // lists of the staged gather, 256 cells per workgroup
    const int32_t *extOff, *extFace;
    const uint16_t* extCell;
    const double *exW, *exMagSf, *exNodc;
};

struct Out {
    double *values, *rhs, *rhs3, *bMat, *bRhs;
};

constexpr int kCells = 256;

template <bool DIV, bool LAP, bool EDIV, int NC, int XE>
__global__ __launch_bounds__(kCells) void k_assemble(MeshIn m, Terms t, Out o) {
    // values kept per face: div its lower and upper coefficient, laplacian one for
    // both sides, the explicit flux
    constexpr int kD = 0, kL = DIV ? 2 : 0, kE = kL + (LAP ? 1 : 0), NV = kE + (EDIV ? 1 : 0);
    constexpr int kMaxUp = gather_max_up(kCells);
    constexpr int kMaxExt = XE == 1 ? gather_max_ext(kCells) : gather_wide_ext();
    constexpr int kMaxLow = gather_max_low(kCells);
    constexpr int kUL = 3;  // own faces per thread and pass
    __shared__ double fU[NV][kMaxUp];
    __shared__ double fE[NV][kMaxExt];
    __shared__ uint16_t exS[kCells], exE[kCells], lowL[kMaxLow][kCells];
    __shared__ int lowN[kCells];
    __shared__ int overflow;
    // the workgroup's rows, one contiguous range of the matrix: written by the cells'
    // threads entry by entry here, and from here with consecutive lanes on
    // consecutive entries (kRows entries fit, 8 per row; more are written directly)
    constexpr int kRows = 8 * kCells;
    __shared__ double rows[kRows];
    const int tid = (int)threadIdx.x, lb = brick_of((int)blockIdx.x, m.run);
    if (lb >= m.nBlocks) return;
    const int c0 = lb * kCells, c1 = min(c0 + kCells, m.N), c = c0 + tid;
    const int fs = m.ownStart[c0], nF = m.ownStart[c1] - fs;
    const int e0 = m.extOff[lb], e1 = m.extOff[lb + 1];
    const bool fits = nF <= kMaxUp && e1 - e0 <= kMaxExt;
    // cell inputs, in flight during phase 1
    const int cc = min(c, c1 - 1);
    const double vol = m.V[cc];
    const int row = m.rowOffs[cc], u0 = m.ownStart[cc], u1 = m.ownStart[cc + 1];
    const int b0 = m.bOff[cc], b1 = m.bOff[cc + 1];
    double told[NC];
#pragma unroll
    for (int k = 0; k < NC; ++k) told[k] = t.Told ? t.Told[(int64_t)NC * cc + k] : 0.0;
    const double src = t.source ? t.source[cc] : 0.0;

    struct In {
        double w, phi, gamma, magSf, nodc, ephi;
    };
    auto load = [&](int f) {
        In a{};
        if (DIV) {
            a.phi = t.phi[f];
            if (t.scheme == FV_LINEAR) a.w = m.w[f];
        }
        if (LAP) {
            a.gamma = t.gamma[f];
            a.magSf = m.magSf[f];
            a.nodc = m.nodc[f];
        }
        if (EDIV) a.ephi = t.ephi[f];
        return a;
    };
    auto make = [&](const In& a, double (&v)[NV]) {
        if (DIV) {
            const double lam = t.scheme == FV_LINEAR ? a.w : (a.phi >= 0.0 ? 1.0 : 0.0);
            v[kD] = -lam * a.phi;          // lower: the neighbour's row, owner's column
            v[kD + 1] = v[kD] + a.phi;     // upper
        }
        if (LAP) v[kL] = a.nodc * (a.gamma * a.magSf);
        if (EDIV) v[kE] = a.ephi;
    };
    auto eload = [&](int k, int f) {
        In a{};
        if (DIV) {
            a.phi = t.phi[f];
            if (t.scheme == FV_LINEAR) a.w = m.exW[k];
        }
        if (LAP) {
            a.gamma = t.gamma[f];
            a.magSf = m.exMagSf[k];
            a.nodc = m.exNodc[k];
        }
        if (EDIV) a.ephi = t.ephi[f];
        return a;
    };
    auto eput = [&](int k, int cl, int cp, int cn, const In& a) {
        double v[NV];
        make(a, v);
#pragma unroll
        for (int j = 0; j < NV; ++j) fE[j][k - e0] = v[j];
        if (k == e0 || cp != cl) exS[cl] = (uint16_t)(k - e0);
        if (k == e1 - 1 || cn != cl) exE[cl] = (uint16_t)(k - e0 + 1);
    };
    // the list records and the first pass's faces are loaded before the barrier
    int ef[XE], ec[XE], ep[XE], en[XE];
#pragma unroll
    for (int x = 0; x < XE; ++x) {
        const int k = min(e0 + tid + x * kCells, e1);  // at most the zero record past the lists
        ef[x] = m.extFace[k];
        ec[x] = m.extCell[k];
        ep[x] = m.extCell[max(k - 1, e0)];
        en[x] = m.extCell[max(min(k + 1, e1 - 1), e0)];
    }
    const int nUp = fits ? nF : 0;
    int nn[kUL];
    In fin[kUL];
    auto own_load = [&](int i0) {
#pragma unroll
        for (int q = 0; q < kUL; ++q) nn[q] = m.nbr[fs + min(i0 + q * kCells, nUp - 1)];
#pragma unroll
        for (int q = 0; q < kUL; ++q) fin[q] = load(fs + min(i0 + q * kCells, nUp - 1));
    };
    auto own_put = [&](int i0) {
#pragma unroll
        for (int q = 0; q < kUL; ++q) {
            const int i = i0 + q * kCells;
            if (i >= nUp) break;
            double v[NV];
            make(fin[q], v);
#pragma unroll
            for (int j = 0; j < NV; ++j) fU[j][i] = v[j];
            if (nn[q] < c1) {
                const int nl = nn[q] - c0;
                const int s = atomicAdd(&lowN[nl], 1);
                if (s < kMaxLow)
                    lowL[s][nl] = (uint16_t)i;
                else
                    overflow = 1;
            }
        }
    };
    if (nUp > 0) own_load(tid);
    In ein[XE];
#pragma unroll
    for (int x = 0; x < XE; ++x)
        if (fits && e0 + tid + x * kCells < e1) ein[x] = eload(e0 + tid + x * kCells, ef[x]);
    exS[tid] = exE[tid] = 0;
    lowN[tid] = 0;
    if (tid == 0) overflow = fits ? 0 : 1;
    __syncthreads();
    if (fits) {
#pragma unroll
        for (int x = 0; x < XE; ++x)
            if (e0 + tid + x * kCells < e1)
                eput(e0 + tid + x * kCells, ec[x], ep[x], en[x], ein[x]);
        own_put(tid);
        for (int i0 = tid + kUL * kCells; i0 < nUp; i0 += kUL * kCells) {
            own_load(i0);
            own_put(i0);
        }
        if (XE > 1)
            for (int k = e0 + tid + XE * kCells; k < e1; k += kCells)
                eput(k, m.extCell[k], m.extCell[max(k - 1, e0)], m.extCell[min(k + 1, e1 - 1)],
                     eload(k, m.extFace[k]));
    }
    const int rbase = m.rowOffs[c0], rn = m.rowOffs[c1] - rbase;
    const bool staged = rn <= kRows;
    __syncthreads();
    if (c < c1) {

    double dDiv = 0.0, dLap = 0.0, acc = 0.0, bDiv[NC], bLap[NC];
#pragma unroll
    for (int k = 0; k < NC; ++k) bDiv[k] = bLap[k] = 0.0;
    double* out = staged ? rows + (row - rbase) : o.values + row;
    auto entry = [&](double cd, double cl) {
        double x = 0.0;
        if (DIV) x += t.cDiv * cd;
        if (LAP) x += t.cLap * cl;
        *out++ = x;
    };
    auto lower = [&](const double (&v)[NV]) {  // this cell is the face's neighbour
        entry(DIV ? v[kD] : 0.0, LAP ? v[kL] : 0.0);
        if (DIV) dDiv -= v[kD + 1];
        if (LAP) dLap -= v[kL];
        if (EDIV) acc -= v[kE];
    };
    auto upper = [&](const double (&v)[NV]) {
        entry(DIV ? v[kD + 1] : 0.0, LAP ? v[kL] : 0.0);
        if (DIV) dDiv -= v[kD];
        if (LAP) dLap -= v[kL];
        if (EDIV) acc += v[kE];
    };
    double* diag;
    if (!overflow) {
        double v[NV];
        for (int k = exS[tid]; k < exE[tid]; ++k) {
#pragma unroll
            for (int j = 0; j < NV; ++j) v[j] = fE[j][k];
            lower(v);
        }
        // the inner lower faces arrived in any order: sorted in registers
        const int n = lowN[tid];
        uint16_t key[kMaxLow];
#pragma unroll
        for (int a = 0; a < kMaxLow; ++a) key[a] = a < n ? lowL[a][tid] : uint16_t(0xFFFF);
        sort_keys<kMaxLow>(key);
#pragma unroll
        for (int a = 0; a < kMaxLow; ++a)
            if (a < n) {
#pragma unroll
                for (int j = 0; j < NV; ++j) v[j] = fU[j][key[a]];
                lower(v);
            }
        diag = out++;
        for (int i = u0 - fs; i < u1 - fs; ++i) {
#pragma unroll
            for (int j = 0; j < NV; ++j) v[j] = fU[j][i];
            upper(v);
        }
    } else {
        double v[NV];
        for (int k = m.lowOff[c]; k < m.lowOff[c + 1]; ++k) {
            make(load(m.lowFace[k]), v);
            lower(v);
        }
        diag = out++;
        for (int f = u0; f < u1; ++f) {
            make(load(f), v);
            upper(v);
        }
    }
    for (int k = b0; k < b1; ++k) {
        const int b = m.bFace[k];
        const bool grad = (DIV || LAP) && t.kind[b] == FV_BC_FIXED_GRADIENT;
        const double d = m.dcb[b];
        double x[NC];  // the face's boundary gradient or value
#pragma unroll
        for (int q = 0; q < NC; ++q)
            x[q] = !grad ? t.Tb[(int64_t)NC * b + q] : t.Tg ? t.Tg[(int64_t)NC * b + q] : 0.0;
        if (DIV) {
            const double pf = t.phi[m.F + b];
            if (grad) dDiv += pf;
#pragma unroll
            for (int q = 0; q < NC; ++q) bDiv[q] -= grad ? pf * (x[q] / d) : pf * x[q];
        }
        if (LAP) {
            const double gm = t.gamma[m.F + b] * m.magSfb[b];
            const double ic = gm * d;
            if (!grad) dLap -= ic;
#pragma unroll
            for (int q = 0; q < NC; ++q) bLap[q] -= grad ? gm * x[q] : ic * x[q];
            o.bMat[b] = grad ? 0.0 : t.cLap * ic;
            o.bRhs[b] = t.cLap * (grad ? gm * x[0] : ic * x[0]);
        } else {
            o.bMat[b] = 0.0;
            o.bRhs[b] = 0.0;
        }
        if (EDIV) acc += t.ephi[m.F + b];
    }
    double dv = 0.0;
    if (t.Told) dv += t.cDdt * (t.rdt * vol);
    if (DIV) dv += t.cDiv * dDiv;
    if (LAP) dv += t.cLap * dLap;
    if (t.source) dv += t.cSource * (src * vol);
    *diag = dv;
#pragma unroll
    for (int q = 0; q < NC; ++q) {
        double r = 0.0;
        if (t.Told) r += t.cDdt * ((t.rdt * told[q]) * vol);
        if (DIV) r += t.cDiv * bDiv[q];
        if (LAP) r += t.cLap * bLap[q];
        if (EDIV) r -= t.cEdiv * ((acc / vol) * vol);
        if (q == 0) o.rhs[c] = r;
        if (NC > 1) o.rhs3[(int64_t)NC * c + q] = r;
    }
    }
    if (!staged) return;
    __syncthreads();
    for (int i = tid; i < rn; i += kCells) o.values[rbase + i] = rows[i];
}

}  // namespace

extern "C" int fv_assemble_terms(fv_linsys* ls, const fv_term* terms, int n, int ncomp,
                                 void* d_rhs3, int* done) {
    return guarded([&] {
        FV_REQUIRE(ls && ls->sp && ls->sp->mesh && done && (terms || n == 0) && n >= 0,
                   "NULL argument");
        FV_REQUIRE(ncomp == 1 || (ncomp == 3 && d_rhs3), "one component, or three with their rhs");
        *done = 0;
        fv_mesh* m = ls->sp->mesh;
        // ddt, div, laplacian, source, explicit div in this order, each at most once, a
        // div or laplacian among them (the order the terms are added in), and faces in
        // upper-triangular order; anything else is assembled term by term
        if (!m->upperTri) return;
        Terms t{};
        const fv_bc* bc = nullptr;
        int last = -1;
        for (int i = 0; i < n; ++i) {
            const fv_term& a = terms[i];
            if (a.kind <= last || a.kind > FV_TERM_EXPLICIT_DIV) return;
            last = a.kind;
            FV_REQUIRE(a.kind >= 0 && a.field, "bad term");
            const double* f = (const double*)a.field;
            if (a.kind == FV_TERM_DDT_EULER) {
                FV_REQUIRE(a.dt > 0.0, "bad ddt arguments");
                t.Told = f;
                t.rdt = 1.0 / a.dt;
                t.cDdt = a.coeff;
            } else if (a.kind == FV_TERM_SOURCE) {
                t.source = f;
                t.cSource = a.coeff;
            } else if (a.kind == FV_TERM_EXPLICIT_DIV) {
                t.ephi = f;
                t.cEdiv = a.coeff;
            } else {
                FV_REQUIRE(a.bc && a.bc->mesh == m, "boundary conditions belong to another mesh");
                FV_REQUIRE(a.d_Tb || m->nB == 0, "NULL field");
                // one boundary condition, one set of boundary values for both terms
                if (bc && (bc != a.bc || t.Tb != a.d_Tb || t.Tg != a.d_Tg)) return;
                bc = a.bc;
                t.kind = a.bc->faceKind.p;
                t.Tb = (const double*)a.d_Tb;
                t.Tg = (const double*)a.d_Tg;
                if (a.kind == FV_TERM_DIV) {
                    FV_REQUIRE(a.scheme == FV_LINEAR || a.scheme == FV_UPWIND, "unknown scheme");
                    t.phi = f;
                    t.scheme = a.scheme;
                    t.cDiv = a.coeff;
                } else {
                    t.gamma = f;
                    t.cLap = a.coeff;
                }
            }
        }
        const bool div = t.phi, lap = t.gamma, ediv = t.ephi;
        if (!(div || lap) || (ediv && (div || ncomp > 1))) return;
        const GatherLists& L = gather_lists(m, kCells);
        const fv_sparsity* sp = ls->sp;
        const MeshIn in{m->nCells,   m->nInt,     (int)L.nBlocks, m->gatherRun, m->nbr.p,   m->ownStart.p,
                        m->lowOff.p, m->lowFace.p, m->bOff.p,     m->bFace.p, sp->rowOffs.p,
                        m->V.p,      m->w.p,       m->magSf.p,    m->nodc.p,  m->magSfb.p,
                        m->dcb.p,    L.extOff.p,   L.extFace.p,   L.extCell.p, L.exW.p,
                        L.exMagSf.p, L.exNodc.p};
        const Out out{ls->values.p, ls->rhs.p, (double*)d_rhs3, ls->bMat.p, ls->bRhs.p};
        hipStream_t s = m->ctx->stream;
        const bool wide = gather_wide(L);
        auto launch = [&](auto D, auto Lp, auto E, auto C) {
            constexpr bool kDiv = decltype(D)::value, kLap = decltype(Lp)::value,
                           kEd = decltype(E)::value;
            constexpr int kC = decltype(C)::value;
            if (wide)
                k_assemble<kDiv, kLap, kEd, kC, 2><<<gather_grid(in.nBlocks, in.run), kCells, 0, s>>>(in, t, out);
            else
                k_assemble<kDiv, kLap, kEd, kC, 1><<<gather_grid(in.nBlocks, in.run), kCells, 0, s>>>(in, t, out);
        };
        using Y = std::true_type;
        using X = std::false_type;
        using C1 = std::integral_constant<int, 1>;
        using C3 = std::integral_constant<int, 3>;
        if (ncomp == 1) {
            if (div && lap) launch(Y{}, Y{}, X{}, C1{});
            else if (div) launch(Y{}, X{}, X{}, C1{});
            else if (ediv) launch(X{}, Y{}, Y{}, C1{});
            else launch(X{}, Y{}, X{}, C1{});
        } else {
            if (div && lap) launch(Y{}, Y{}, X{}, C3{});
            else if (div) launch(Y{}, X{}, X{}, C3{});
            else launch(X{}, Y{}, X{}, C3{});
        }
        FV_LAUNCH_CHECK();
        *done = 1;
    });
}
