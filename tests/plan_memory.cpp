// plan_memory.cpp -- the library's set-up on host memory: hipMalloc and the other runtime calls a
// set-up makes are defined here (the program's definitions come before the runtime's), so that an
// allocation can be made to fail and every buffer's size, fill and content can be looked at
// without a GPU.  Nothing is launched.  test_plan_memory.py builds and runs it:
//   plan_memory CHECK [args]  prints what is wrong, or "ok"
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <string>
#include <vector>

#include "mbgpu_internal.h"

namespace {

struct Block {
    size_t size;
    bool filled;                       // 0xff bytes were once set over all of it
};
std::map<const void*, Block> live;
long nalloc = 0, nfree = 0, fail_at = -1;   // allocations made, frees, the allocation that fails
hipError_t last = hipSuccess;               // the runtime's last error, kept until it is asked for
int wrong = 0;

}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t n)
{
    *p = nullptr;
    if (nalloc++ == fail_at) return last = hipErrorOutOfMemory;
    *p = calloc(n, 1);
    live[*p] = Block{n, false};
    return hipSuccess;
}
hipError_t hipFree(void* p)
{
    if (!live.erase(p)) {
        printf("free of a block that is not live\n");
        ++wrong;
        return hipErrorInvalidValue;
    }
    ++nfree;
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned int)
{
    *p = calloc(n, 1);
    return hipSuccess;
}
hipError_t hipHostFree(void* p)
{
    free(p);
    return hipSuccess;
}
hipError_t hipMemset(void* p, int v, size_t n)
{
    memset(p, v, n);
    auto b = live.find(p);
    if (b != live.end() && b->second.size == n && v == 0xff) b->second.filled = true;
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind)
{
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t)
{
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError(void)
{
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamCreate(hipStream_t* s)
{
    *s = nullptr;
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned int)
{
    *s = nullptr;
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e)
{
    *e = nullptr;
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n)
{
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetDevice(int* d)
{
    *d = 0;
    return hipSuccess;
}
}

namespace {

void check(bool ok, const std::string& what)
{
    if (ok) return;
    printf("%s\n", what.c_str());
    ++wrong;
}

size_t size_of(const void* p)
{
    auto b = live.find(p);
    return b == live.end() ? 0 : b->second.size;
}

// ------------------------------------------------------------------ electrostatics ----
struct Call {
    const char* name;
    int nw, imcon;
    double L, alpha, rcut;
    int kmax[3], recip;
};
const Call calls[] = {
    {"box", 8, 1, 12.0, 0.55, 1.1, {8, 8, 8}, 0},         // (short cut-offs: short tables)
    {"other cell", 8, 1, 13.0, 0.55, 1.1, {8, 8, 8}, 0},
    {"other k list", 8, 2, 12.0, 0.5, 1.0, {11, 9, 17}, 0},
    {"mesh", 8, 1, 12.0, 0.6, 1.1, {8, 8, 8}, 1},
    {"cluster", 8, 0, 3.0, 0.0, 3.0, {1, 1, 1}, 0},
    {"other size", 9, 1, 12.0, 0.55, 1.1, {8, 8, 8}, 0},
};
constexpr int NCALLS = sizeof calls / sizeof calls[0];

int configure(ElecState& S, const Call& c)
{
    mbgpu_elec_params p = {};
    p.rcut = c.rcut;
    p.alpha = c.alpha;
    for (int i = 0; i < 3; ++i) p.kmax[i] = c.kmax[i];
    p.toler = 1e-12;
    p.omega = 0.3;
    p.max_iter = 100;
    p.gamma = 0.4267;
    p.polr[0] = p.polr[2] = p.polr2[0] = 1.31;
    p.polr[1] = p.polr2[1] = 0.294;
    p.athole = p.athole13 = 0.055;
    p.athole12 = 0.626;
    p.ascc = p.ascd = 0.4;
    CellGeom g = {};
    g.imcon = c.imcon;
    const double cell[9] = {c.L, 0, 0, 0, c.L, 0, 0, 0, c.imcon == 2 ? c.L + 1.0 : c.L};
    for (int i = 0; i < 9; ++i) g.c[i] = cell[i];
    S.recip = c.recip;
    S.sp_order = 6;
    for (int i = 0; i < 3; ++i) S.sp_grid[i] = 16;
    std::string err;
    return elec_configure(S, c.nw, g, cell, &p, err);
}

// every buffer that an evaluation after a successful configure reads or writes is there, as large
// as the launch parameters say, and holds what a new state's holds (R)
void complete(const ElecState& S, const ElecState& R, const Call& c, const std::string& when)
{
    const ElecBuffers &E = S.E, &F = R.E;
    const ElecDev& P = S.P;
    const size_t n = 4 * c.nw, nr = 3 * c.nw;
    auto need = [&](const char* name, const void* p, size_t bytes) {
        check(size_of(p) >= bytes, when + ": " + name + " holds " + std::to_string(size_of(p)) + " of " +
                                       std::to_string(bytes) + " bytes");
    };
    auto same = [&](const char* name, const void* p, const void* q, size_t bytes) {
        need(name, p, bytes);
        if (size_of(p) >= bytes) check(memcmp(p, q, bytes) == 0, when + ": " + name + " is another plan's");
    };
#define NEED(f, count) need(#f, E.f, sizeof(*E.f) * (size_t)(count))
#define SAME(f, count) same(#f, E.f, F.f, sizeof(*E.f) * (size_t)(count))
    check(P.n == (int)n && P.K == R.P.K && P.nrun == R.P.nrun && P.rvolm == R.P.rvolm && P.drewd == R.P.drewd &&
              P.kchunks == R.P.kchunks && P.fchunks == R.P.fchunks && P.rpc == R.P.rpc,
          when + ": launch parameters of another plan");
    NEED(x, n); NEED(y, n); NEED(z, n); NEED(chge, n); NEED(dg, 6 * c.nw); NEED(tin, 36 * c.nw);
    NEED(cntA, n); NEED(cntP, n); NEED(dip, 3 * n); NEED(dip0, 3 * n); NEED(efk, 3 * n); NEED(emu, 3 * n);
    NEED(efdc, 3 * n); NEED(efdd, 3 * n); NEED(cg_p, nr * 3); NEED(cg_q, nr * 3); NEED(cg_r, nr * 3);
    NEED(cg_z, nr * 3); NEED(cg_u, nr * 3); NEED(cg_w, nr * 3); NEED(cg_m, nr * 3); NEED(cg_s, nr * 3);
    NEED(cg_tmu, nr * 3); NEED(cg_minv, 45 * c.nw); NEED(cgblk, 5 * ((c.nw + 6) / 7)); NEED(ksum, 15 * n);
    NEED(state, 16); NEED(vr, n); NEED(vdcr, n); NEED(vesp, n); NEED(f2, 3 * n); NEED(fsite, 3 * n); NEED(e1, n);
    NEED(e2, n); NEED(w2, 9 * n); NEED(fmsum, 3 * n); NEED(fmx, 9 * n); NEED(eout, nr); NEED(wout, 9 * nr);
    NEED(sout, 9 * nr); NEED(scal, 41); NEED(err, 4); NEED(pk, EL_PK_N);
    check(P.capA > 0 && P.capP > 0, when + ": no neighbour rows");
    NEED(nbrA, n * P.capA); NEED(nbrP, n * P.capP); NEED(tens, n * P.capP);
    const int nkb = c.imcon == 0 ? 0 : std::max((P.K + 63) / 64, P.n / 4);
    NEED(blk, 8 * nkb + 8 * n + 24 * ((c.nw + 15) / 16));
    NEED(Fpart, std::max(c.imcon ? 16 * P.kchunks : 0, 6 * P.fchunks) * n);
    SAME(tab, 4 * (F.ntab + 1));
    if (c.imcon == 0) return;
    const RsPlan& Q = P.rs;
    check(Q.ng == R.P.rs.ng && Q.ntiles == R.P.rs.ntiles && Q.kt == R.P.rs.kt && Q.nch == R.P.rs.nch &&
              Q.pair == E.rs_pair && Q.ak == E.rs_ak && Q.kpos == E.rs_kpos,
          when + ": matrix passes of another plan");
    SAME(kv, 8 * P.K); SAME(runs, 4 * P.nrun); SAME(runk, P.nrun); NEED(kf, 16 * P.K);
    SAME(rs_pair, 16 * Q.ng); SAME(rs_ak, 16 * Q.ng * (8 * Q.ntiles + 1)); SAME(rs_kpos, P.K);
    NEED(pht, (n + RS_PAD) * Q.kt); NEED(Spart, 4 * std::max(Q.nch, Q.nchq) * Q.ng * RS_SLOT(Q.ntiles));
    NEED(phc, 3 * P.kstride * n); NEED(phs, 3 * P.kstride * n);
    check(P.kstride > std::max({P.km[0], P.km[1], P.km[2]}), when + ": phase tables too short");
    if (c.recip) check(S.sp && S.spg, when + ": no particle mesh");
#undef NEED
#undef SAME
}

// A, then B with its k-th allocation failing, then A and B again
void elec_failures()
{
    for (int a = -1; a < NCALLS; ++a)
        for (int b = 0; b < NCALLS; ++b)
            for (long k = 0;; ++k) {
                ElecState S, RA, RB;
                const std::string when = std::string(a < 0 ? "new state" : calls[a].name) + ", then " + calls[b].name +
                                         " without allocation " + std::to_string(k);
                fail_at = -1;
                check(configure(RB, calls[b]) == 0, when + ": reference refused");
                if (a >= 0) {
                    check(configure(RA, calls[a]) == 0, when + ": reference refused");
                    check(configure(S, calls[a]) == 0, when + ": first call refused");
                }
                fail_at = nalloc + k;
                const int rc = configure(S, calls[b]);
                const bool reached = nalloc > fail_at;
                fail_at = -1;
                check((rc != 0) == reached, when + ": returned " + std::to_string(rc));
                check(hipGetLastError() == hipSuccess, when + ": the error is left to the next launch");
                if (a >= 0) {
                    check(configure(S, calls[a]) == 0, when + ": the call that follows is refused");
                    complete(S, RA, calls[a], when + ", then " + calls[a].name);
                }
                check(configure(S, calls[b]) == 0, when + ": the repeated call is refused");
                complete(S, RB, calls[b], when + ", repeated");
                elec_release(S);
                elec_release(RA);
                elec_release(RB);
                if (!reached) break;
            }
    check(live.empty(), std::to_string(live.size()) + " blocks left");
}

// A call with the parameters of the one before frees and allocates nothing.
void elec_repeats()
{
    for (int a = -1; a < NCALLS; ++a)
        for (int b = 0; b < NCALLS; ++b) {
            ElecState S;
            const std::string when = std::string(a < 0 ? "new state" : calls[a].name) + ", then " + calls[b].name;
            if (a >= 0) check(configure(S, calls[a]) == 0, when + ": first call refused");
            check(configure(S, calls[b]) == 0, when + ": refused");
            std::vector<unsigned char> key, key2;
            elec_key_append(S, 1, 1, 10, key);
            const long n0 = nalloc, f0 = nfree;
            check(configure(S, calls[b]) == 0, when + ": refused again");
            elec_key_append(S, 1, 1, 10, key2);
            check(nalloc == n0 && nfree == f0, when + ": " + std::to_string(nalloc - n0) + " allocations and " +
                                                  std::to_string(nfree - f0) + " frees in a repeated call");
            check(key == key2, when + ": a repeated call has another graph key");
            elec_release(S);
        }
}

// MBGPU_POISON=1 (set by the caller): every buffer but the integer ones is filled when it is made.
void elec_poison()
{
    for (const Call& c : calls) {
        ElecState S;
        check(configure(S, c) == 0, std::string(c.name) + ": refused");
        const ElecBuffers& E = S.E;
        std::set<const void*> ints = {E.cntA, E.cntP, E.nbrA, E.nbrP, E.err, E.runs, E.runk, E.rs_pair, E.rs_kpos,
                                      S.cells.key, S.cells.sidx, S.cells.start};
        if (S.sp) ints.insert({S.sp->gi, S.sp->bin_off, S.sp->bin_site, S.sp->flag});
        const std::map<const void*, const char*> names = {{E.tens, "tens"}, {E.pht, "pht"}, {E.rs_ak, "rs_ak"}};
        for (auto& b : live) {
            auto n = names.find(b.first);
            check(b.second.filled || ints.count(b.first),
                  std::string(c.name) + ": " + (n == names.end() ? "a buffer" : n->second) + " of " +
                      std::to_string(b.second.size) + " bytes is not filled");
        }
        elec_release(S);
    }
}

// Prints the bytes of the neighbour rows of a cluster of nw waters, every pair within rcut.
void cluster_rows(int nw)
{
    ElecState S;
    const Call c = {"cluster", nw, 0, 40.0, 0.0, 40.0, {1, 1, 1}, 0};
    check(configure(S, c) == 0, "refused");
    printf("%zu\n", size_of(S.E.nbrA) + size_of(S.E.nbrP) + size_of(S.E.tens));
    elec_release(S);
}

// ----------------------------------------------- water terms, MB-pol (and its precisions) ----
int configure_water(WaterState& S, double rcut)
{
    mbgpu_water_params p = {};
    p.rcut = p.rvdw = rcut;
    for (int t = 0; t < 3; ++t) {
        p.c6[t] = 1000.0;
        p.a6[t] = p.a8[t] = 9.0;
    }
    p.dispersion = p.ps_monomer = 1;
    CellGeom g = {};
    g.imcon = 1;
    const double cell[9] = {12, 0, 0, 0, 12, 0, 0, 0, 12};
    std::string err;
    return water_configure(S, 8, g, cell, &p, nullptr, err);
}

void water_failures()
{
    const double cut[2] = {1.0, 1.5};
    for (int first = 0; first < 2; ++first)
        for (long k = 0;; ++k) {
            WaterState S;
            const std::string when = std::string(first ? "second" : "first") + " cut-off without allocation " +
                                     std::to_string(k);
            if (first) check(configure_water(S, cut[0]) == 0, when + ": first call refused");
            fail_at = nalloc + k;
            const int rc = configure_water(S, cut[first]);
            const bool reached = nalloc > fail_at;
            fail_at = -1;
            check((rc != 0) == reached, when + ": returned " + std::to_string(rc));
            for (int again = 0; again < 2; ++again) {
                check(configure_water(S, cut[again]) == 0, when + ": a call that follows is refused");
                const size_t table = sizeof(double) * 3 * S.P.ngrid, nr = 24;
                check(S.P.ngrid == (int)(cut[again] / 0.0001 + 0.5) + 7 && size_of(S.B.vvv) == table &&
                          size_of(S.B.ggg) == table,
                      when + ": tables of " + std::to_string(size_of(S.B.vvv)) + " and " +
                          std::to_string(size_of(S.B.ggg)) + " bytes, not " + std::to_string(table));
                check(size_of(S.B.mono) == 13 * nr * 8 && size_of(S.B.wsc) && size_of(S.B.asc) && size_of(S.B.fw) &&
                          size_of(S.B.eout) && size_of(S.B.wout) && size_of(S.B.psc) && size_of(S.B.pcm) &&
                          size_of(S.B.pidx) && size_of(S.B.pidxm) && size_of(S.B.scal),
                      when + ": a buffer is missing");
            }
            water_release(S);
            if (!reached) break;
        }
    check(live.empty(), std::to_string(live.size()) + " blocks left");
}

int mbpol(mbgpu_ctx* c)
{
    const double cell[9] = {12, 0, 0, 0, 12, 0, 0, 0, 12};
    const int list[6] = {1, 2, 3, 4, 5, 6};
    double x[8] = {}, f[8] = {}, e = 0.0, v = 0.0, s[9] = {};
    return mbgpu_mbpol_forces(c, 1, cell, 6, list, x, x, x, f, f, f, &e, &v, s);
}

std::multiset<size_t> sizes()
{
    std::multiset<size_t> r;
    for (auto& b : live) r.insert(b.second.size);
    return r;
}

// MB-pol's cluster buffers, first in FP64 and then with the FP32 polynomials: whatever fails, the
// calls that follow hold the same buffers as in a context where nothing failed
void mbpol_failures()
{
    for (int step = 0; step < 3; ++step) {
        // 0: the first evaluation, 1: the change of precision after it, 2: before it
        auto call = [&](mbgpu_ctx* c, int s) { return s == 0 ? mbpol(c) : mbgpu_set_precision(c, 3); };
        std::multiset<size_t> want;
        for (long k = -1;; ++k) {
            const std::string when = "MB-pol, step " + std::to_string(step) + " without allocation " + std::to_string(k);
            mbgpu_ctx* c = mbgpu_create(2, 8);
            if (step == 1) check(mbpol(c) == 0, when + ": evaluation refused");
            fail_at = k < 0 ? -1 : nalloc + k;
            const int rc = call(c, step);
            const bool reached = k >= 0 && nalloc > fail_at;
            fail_at = -1;
            check((rc != 0) == reached, when + ": returned " + std::to_string(rc));
            check(mbpol(c) == 0, when + ": the evaluation that follows is refused");
            if (step) check(mbgpu_set_precision(c, 3) == 0, when + ": the precision is refused again");
            check(mbpol(c) == 0, when + ": the last evaluation is refused");
            if (k < 0) want = sizes();
            else check(sizes() == want, when + ": " + std::to_string(live.size()) + " buffers, not the " +
                                            std::to_string(want.size()) + " of an undisturbed context");
            mbgpu_destroy(c);
            check(live.empty(), when + ": blocks left");
            if (k >= 0 && !reached) break;
        }
    }
}

}  // namespace

int main(int argc, char** argv)
{
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "elec_failures") elec_failures();
    else if (what == "elec_repeats") elec_repeats();
    else if (what == "elec_poison") elec_poison();
    else if (what == "cluster_rows" && argc > 2) cluster_rows(atoi(argv[2]));
    else if (what == "water_failures") water_failures();
    else if (what == "mbpol_failures") mbpol_failures();
    else check(false, "no such check: " + what);
    if (!wrong) printf("ok\n");
    return wrong != 0;
}
