// The server's worker over a stand-in device and solver: which sectors and engines it builds, keeps and gives up
// under a budget.  Usage: server_host <scenario>; exit status 0, or a message and 3.
#include "device_stub.hpp"

#include <cmath>
#include <string>
#include <tuple>

#include "bh_engine.hpp"
#include "bh_internal.hpp"

namespace {

size_t ham_bytes_per_state = 100, engine_bytes = 1000;
bool accept_mixed = true, fullre = true;
int hams_built = 0;

// every lane is done after its first chunk; its levels are J, J + 1, ...
class Engine final : public LzEngineBase {
    std::vector<double> J;
    std::vector<char> on;
    bool f64;

   public:
    Engine(int B, bool d) : J(B, 0.0), on(B, 0), f64(d) { stub::live.insert(this); }
    ~Engine() override { stub::check(stub::live.erase(this) == 1, "engine destroyed twice"); }
    void alive() const { stub::check(stub::live.count(this) == 1, "call of a released engine"); }
    int admit(int s, double j, double) override {
        alive();
        J[s] = j;
        on[s] = 1;
        return BH_OK;
    }
    int run(int) override {
        alive();
        return BH_OK;
    }
    int check(std::vector<int>& fin) override {
        alive();
        for (size_t i = 0; i < on.size(); ++i)
            if (on[i]) {
                on[i] = 0;
                fin.push_back(static_cast<int>(i));
            }
        return BH_OK;
    }
    int finish(const std::vector<int>& lanes, std::vector<LaneResult>& out, bool) override {
        alive();
        for (int l : lanes) {
            LaneResult r;
            for (int i = 0; i < 4; ++i) r.evals.push_back(J[l] + i);
            r.resid.assign(4, 0.0);
            r.errest.assign(4, 0.0);
            r.iters = 1;
            r.status = BH_OK;
            out.push_back(r);
        }
        return BH_OK;
    }
    int lanes() const override { return static_cast<int>(on.size()); }
    int active() const override {
        alive();
        int n = 0;
        for (char c : on) n += c;
        return n;
    }
    int steps_of(int) const override { return 1; }
    int suggest_chunk() const override { return 1; }
    size_t device_bytes() const override { return engine_bytes; }
    bool fp64() const override { return f64; }
    int export_tridiag(int, double*, double*, double*) override { return BH_EINVAL; }
    void set_deflation_barrier(bool) override {}
};

}  // namespace

int bh_set_error(const bh_ctx*, int code, const std::string&) { return code; }
int64_t bh_binom_host(int n, int k) {
    double r = 1;
    for (int i = 1; i <= k; ++i) r = r * (n - k + i) / i;
    return static_cast<int64_t>(std::llround(r));
}
std::unique_ptr<LzEngineBase> bh_make_engine(bh_ctx*, bh_ham* h, int prec, int B, const bh_lanczos_opts&, hipStream_t, bool,
                                             int* rc) {
    stub::check(stub::live.count(h) == 1, "engine over a released Hamiltonian");
    *rc = BH_OK;
    return std::make_unique<Engine>(B, prec == BH_PREC_FP64);
}
size_t bh_engine_bytes(int64_t, int, int, const bh_lanczos_opts&) { return engine_bytes; }
bool bh_lz_fullre(int64_t, const bh_lanczos_opts&) { return fullre; }
bool bh_lane_accepted(int, const double*, const double*, int, double) {
    if (accept_mixed) return true;
    accept_mixed = true;  // the next one is the rerun
    return false;
}
bh_lanczos_opts bh_fallback_opts(const bh_lanczos_opts& o) { return o; }
bh_lanczos_opts bh_fallback_full_opts(const bh_lanczos_opts& o) { return o; }

extern "C" {

int bh_ctx_create(int, size_t budget, bh_ctx** out) {
    *out = new bh_ctx();
    (*out)->budget = budget;
    return BH_OK;
}
int bh_ctx_destroy(bh_ctx* c) {
    delete c;
    return BH_OK;
}
int bh_lattice_neighbours(int, int Lx, int Ly, int, int* off, int*) {
    for (int i = 0; i <= Lx * Ly; ++i) off[i] = 0;
    return 0;
}
int bh_basis_build(bh_ctx*, int m, int n, int, bh_basis** out) {
    *out = new bh_basis();
    (*out)->D = bh_binom_host(m + n - 1, n);
    stub::live.insert(*out);
    return BH_OK;
}
int bh_basis_destroy(bh_basis* b) {
    stub::check(stub::live.erase(b) == 1, "basis destroyed twice");
    return BH_OK;
}
int bh_hamiltonian_build(bh_ctx*, const bh_basis* b, const int*, const int*, unsigned, bh_ham** out) {
    stub::check(stub::live.count(b) == 1, "Hamiltonian over a released basis");
    *out = new bh_ham();
    (*out)->D = b->D;
    (*out)->nnz = 10 * b->D;
    stub::live.insert(*out);
    ++hams_built;
    return BH_OK;
}
int bh_ham_destroy(bh_ham* h) {
    stub::check(stub::live.erase(h) == 1, "Hamiltonian destroyed twice");
    return BH_OK;
}
int64_t bh_ham_device_bytes(const bh_ham* h) {
    stub::check(stub::live.count(h) == 1, "bytes of a released Hamiltonian");
    return static_cast<int64_t>(h->D * ham_bytes_per_state);
}
int bh_lanczos(bh_ctx*, bh_ham*, int, const double*, const double*, const bh_lanczos_opts*, bh_lanczos_result*) {
    return BH_EINVAL;
}

}  // extern "C"

static bh_server* server(size_t budget) {
    bh_ctx* ctx = new bh_ctx();
    bh_server_opts o{};
    o.lanes = 4;
    o.hbm_budget = budget;
    o.prec = BH_PREC_MIXED;
    o.lanczos.k = 4;
    bh_server* S = nullptr;
    stub::check(bh_server_create(ctx, &o, &S) == BH_OK, "server");
    return S;
}

static void serve(bh_server* S, int m, int n, double J, int status) {
    bh_request q{};
    q.Lx = m;
    q.Ly = 1;
    q.n = n;
    q.J = J;
    q.U = 1.0;
    uint64_t id = 0;
    stub::check(bh_server_submit(S, &q, &id) == BH_OK, "submit");
    bh_result r{};
    stub::check(bh_server_wait(S, id, 20.0, &r) == BH_OK, "no answer within 20 s");
    stub::check(r.status == status, "status of a request");
    if (status == BH_OK)
        for (int i = 0; i < 4; ++i) stub::check(r.evals[i] == J + i, "levels of a request");
}

int main(int argc, char** argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "evict") {
        // chains of 4, 5 and 6 sites, four bosons (D = 35, 70, 126): their matrices together are over the budget, so an idle
        // sector is given up whole for another, sectors before and after it in the map's order
        bh_server* S = server(19000);
        for (int round = 0; round < 3; ++round)
            for (int m : {4, 5, 6, 5, 4, 6}) serve(S, m, 4, 0.25 * m + round, BH_OK);
        stub::check(hams_built > 3, "no sector was given up");
        stub::check(bh_server_destroy(S) == BH_OK, "destroy");
        stub::check(stub::live.empty(), "streams or handles left behind");
    } else if (what == "rerun") {
        // a rejected mixed solve under a budget with room for the matrix (3,500 bytes) and two engines, and little more
        accept_mixed = fullre = false;
        bh_server* S = server(6000);
        serve(S, 4, 4, 0.5, BH_OK);
        stub::check(accept_mixed, "no rerun");
        stub::check(bh_server_destroy(S) == BH_OK, "destroy");
    } else {
        stub::fail("unknown scenario");
    }
    std::puts("ok");
    return 0;
}
