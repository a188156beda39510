// host_checks.cpp -- host code of libcismgpu.so on a HIP runtime without a
// device (hip_on_host.h).  Usage: host_checks LIB CHECK; exit status 0 when
// the check holds.
#include "hip_on_host.h"

#include <dlfcn.h>

#include "cismgpu.h"

#define FN(name) static decltype(&name) p_##name
FN(cismgpu_system_create);
FN(cismgpu_system_destroy);
FN(cismgpu_system_set_matrix);
FN(cismgpu_system_assemble_3d);
FN(cismgpu_system_solve);
FN(cismgpu_system_residual);
FN(cismgpu_system_set_x);
FN(cismgpu_system_get_x);
FN(cismgpu_system_internal_stress);

static int bad = 0;
#define EXPECT(c)                                                       \
    do {                                                                \
        if (!(c)) { printf("line %d: not %s\n", __LINE__, #c); ++bad; } \
    } while (0)

// Flat ice on an n x n block of owned vertices, every cell and vertex of the
// inner block active; nothing here is computed, the calls only have to pass.
struct Ice {
    cismgpu_grid g{};
    cismgpu_system* S = nullptr;
    std::vector<double> vert, levels, layers, cells;
    std::vector<int32_t> acell, avert, ocean;
    cismgpu_assembly_in in{};

    Ice(int n, int nz, int bc = 3) {
        g.nx = g.ny = n + 4;
        g.nz = nz;
        g.ilo = g.jlo = 3;
        g.ihi = g.jhi = n + 2;
        g.global_bc = bc;
        const int nv = g.nx - 1;
        vert.assign((size_t)nv * nv, 1.0);
        levels.resize(nz + 1);
        for (int k = 0; k <= nz; ++k) levels[k] = (double)k / nz;
        layers.assign((size_t)(nz - 1) * g.nx * g.ny, 1.0);
        cells.assign((size_t)g.nx * g.ny, 1.0);
        acell.assign(cells.size(), 1);
        avert.assign(vert.size(), 1);
        ocean.assign(cells.size(), 0);
        in.dx = in.dy = 1.0;
        in.sigma = in.stagwbndsigma = levels.data();
        in.active_cell = acell.data();
        in.active_vertex = avert.data();
        for (const double** p : {&in.xVertex, &in.yVertex, &in.stagusrf, &in.stagthck, &in.dusrf_dx, &in.dusrf_dy})
            *p = vert.data();
        in.flwafact = layers.data();
        in.whichefvs = 2;
        in.n_glen = 3.0;
        EXPECT(p_cismgpu_system_create(&g, &S) == 0);
    }
    ~Ice() { p_cismgpu_system_destroy(S); }

    int assemble() { return p_cismgpu_system_assemble_3d(S, &in, nullptr); }
    // the fields of the lateral condition too: a larger input block
    int assemble_lateral() {
        cismgpu_assembly_in b = in;
        b.ocean_mask = ocean.data();
        b.usrf = b.thck = cells.data();
        b.stagusrf_lateral = b.stagthck_lateral = vert.data();
        return p_cismgpu_system_assemble_3d(S, &b, nullptr);
    }
    int solve(int precision = CISMGPU_FP64, int maxiters = 6) {
        onhost::launched.clear();
        cismgpu_solve_opts o{CISMGPU_ALGO_CHRONGEAR, 2, 5, maxiters, 0.0, precision, 1e-4, 2, 0};
        cismgpu_solve_info info;
        return p_cismgpu_system_solve(S, &o, &info);
    }
};

// Scalars that keep a solve going: norms of one, a residual of a half.
static void converging(const std::string& name, void** args) {
    if (name.find("k_scalars") == std::string::npos) return;
    double* scal = *(double**)args[7];
    scal[6] = 1.0;      // L2 norm of the rhs
    scal[8] = 0.5;      // relative residual of a check
    scal[12] = 1.0;     // plain dot product
    if (auto* mirror = *(unsigned long long**)args[9]) {
        memcpy(mirror, &scal[8], 8);
        mirror[1] = 4 * *(unsigned long long*)args[10];
        mirror[2] = mirror[0] ^ mirror[1];
    }
}

// A re-assembly that fails once its inputs are being replaced: the element
// form of the products reads those inputs, so what follows keeps to the rows
// of the old matrix, and the diagnostics, which have nothing else, refuse.
static void failed_reassembly(bool copy_fails) {
    Ice s(8, 3);
    std::vector<double> tau(s.layers.size());
    EXPECT(s.assemble() == 0);
    s.solve();
    EXPECT(onhost::count("k_spmv_elem") > 0);
    if (copy_fails) onhost::copies_to_failure = 5;
    else onhost::fail_malloc = true;
    EXPECT((copy_fails ? s.assemble() : s.assemble_lateral()) != 0);
    onhost::copies_to_failure = -1;
    onhost::fail_malloc = false;
    s.solve();
    EXPECT(onhost::count("k_spmv_elem") == 0 && onhost::count("k_spmv") > 0);
    onhost::launched.clear();
    p_cismgpu_system_residual(s.S, nullptr, nullptr, nullptr, nullptr);
    EXPECT(onhost::count("k_spmv_elem") == 0 && onhost::count("k_spmv") > 0);
    onhost::launched.clear();
    EXPECT(p_cismgpu_system_internal_stress(s.S, tau.data(), nullptr, nullptr, nullptr, nullptr, nullptr) != 0);
    EXPECT(onhost::count("k_internal_stress") == 0);
    EXPECT(s.assemble() == 0);            // an input block of the first size is there again
    s.solve();
    EXPECT(onhost::count("k_spmv_elem") > 0);
    EXPECT(p_cismgpu_system_internal_stress(s.S, tau.data(), nullptr, nullptr, nullptr, nullptr, nullptr) == 0);
}

// The products test for the no-ice halo rule only where it zeroes owned
// columns (rows given by the caller; mode 3).
static void zero_store(int bc, bool expected) {
    Ice s(8, 3, bc);
    const size_t n = s.vert.size() * 3;
    const std::vector<double> A(27 * n), b(n);
    EXPECT(p_cismgpu_system_set_matrix(s.S, s.avert.data(), A.data(), A.data(), A.data(), A.data(), b.data(), b.data(),
                                       0) == 0);
    s.solve();
    EXPECT(onhost::count("k_spmv_sym64ILi3E") == (expected ? 5 : 0));
    EXPECT(onhost::count("k_spmv_sym64ILi1E") == (expected ? 1 : 6));
    EXPECT(s.assemble() == 0);
    s.solve();
    EXPECT(onhost::count("Li3E") == 0);
}

// Levels that a workgroup of a product takes: whole columns where a share would
// be too thin to pay, shares elsewhere; and every partial sum is summed.
static void level_shares(int n, int nz, int half64, int rows16) {
    Ice s(n, nz, 1);
    const size_t m = s.vert.size() * nz;
    std::vector<double> A(27 * m), b(m);
    EXPECT(p_cismgpu_system_set_matrix(s.S, s.avert.data(), A.data(), A.data(), A.data(), A.data(), b.data(), b.data(),
                                       0) == 0);
    const int tiles = (n + 63) / 64 * ((n + 3) / 4);
    int kper = 0, blocks = 0;
    onhost::on_launch = [&](const std::string& name, void** args) {
        if (name.find("k_spmv_sym64") != std::string::npos || name.find("k_spmv_q") != std::string::npos) {
            kper = *(int*)args[9];
            blocks = onhost::grid.x * onhost::grid.y;
            EXPECT((int)onhost::grid.x == tiles && (int)onhost::grid.y == (nz + kper - 1) / kper);
        }
        // the stage of the first iteration takes the product's sums as its second
        if (name.find("k_scalars") != std::string::npos && *(int*)args[0] == 2) EXPECT(*(int*)args[5] == blocks);
        converging(name, args);
    };
    s.solve();
    EXPECT(kper == half64);
    kper = 0;
    s.solve(CISMGPU_MIXED_BF16);
    EXPECT(kper == rows16);
    onhost::on_launch = nullptr;
}

// A solve keeps to the FP32 product it began with, whatever happens to the
// environment meanwhile: the counts of the partial sums belong to it.
static void one_product() {
    Ice s(64, 3);
    EXPECT(s.assemble() == 0);
    for (const char* first : {"1", "0"}) {
        int n = 0;
        setenv("CISMGPU_SPMV_SYMX", first, 1);
        onhost::on_launch = [&](const std::string& name, void** args) {
            setenv("CISMGPU_SPMV_SYMX", ++n % 2 ? "0" : "1", 1);
            converging(name, args);
        };
        s.solve(CISMGPU_MIXED_FP32, 12);
        const int marching = onhost::count("k_spmv_symj"), rereading = onhost::count("k_spmv_symI");
        EXPECT(first[0] == '1' ? marching > 4 && rereading == 0 : marching == 0 && rereading > 4);
    }
    unsetenv("CISMGPU_SPMV_SYMX");
    onhost::on_launch = nullptr;
}

// Large copies in and out, in chunks by several threads: every value arrives,
// also without heap or pinned memory, and a failing copy is reported.
static void large_copies(bool no_heap, bool no_pinned) {
    Ice s(210, 10);
    const size_t n = s.vert.size() * 10;          // 3.6 MB each: a partial last chunk
    std::vector<double> u(n), v(n), a(n), b(n);
    for (size_t i = 0; i < n; ++i) { u[i] = (double)i; v[i] = -(double)i - 0.5; }
    int in = 0, out = 0;
    auto hook = [&](const std::string& name, void** args) {
        if (name.find("k_vec_in") != std::string::npos)
            EXPECT(memcmp(*(double**)args[1], in++ % 2 ? v.data() : u.data(), n * sizeof(double)) == 0);
        if (name.find("k_vec_out") != std::string::npos)
            memcpy(*(double**)args[2], out++ % 2 ? u.data() : v.data(), n * sizeof(double));
    };
    onhost::on_launch = hook;
    onhost::fail_pinned = no_pinned;
    onhost::heap_fails = no_heap;
    const int st_in = p_cismgpu_system_set_x(s.S, u.data(), v.data());
    const int st_out = p_cismgpu_system_get_x(s.S, a.data(), b.data());
    onhost::heap_fails = false;
    EXPECT(st_in == 0 && in == 2 && st_out == 0 && out == 2);
    EXPECT(a == v && b == u);
    onhost::copies_to_failure = 2;
    EXPECT((p_cismgpu_system_get_x(s.S, a.data(), b.data()) != 0) == !no_pinned);   // two whole copies, or many chunks
    onhost::copies_to_failure = -1;
    onhost::on_launch = nullptr;
}

int main(int argc, char** argv) {
    if (argc != 3) return 2;
    void* lib = dlopen(argv[1], RTLD_NOW);
    if (!lib) { printf("%s\n", dlerror()); return 2; }
#define LOAD(name) p_##name = (decltype(p_##name))dlsym(lib, #name)
    LOAD(cismgpu_system_create);
    LOAD(cismgpu_system_destroy);
    LOAD(cismgpu_system_set_matrix);
    LOAD(cismgpu_system_assemble_3d);
    LOAD(cismgpu_system_solve);
    LOAD(cismgpu_system_residual);
    LOAD(cismgpu_system_set_x);
    LOAD(cismgpu_system_get_x);
    LOAD(cismgpu_system_internal_stress);
    const std::map<std::string, std::function<void()>> checks = {
        {"reassembly_out_of_memory", [] { failed_reassembly(false); }},
        {"reassembly_failed_copy", [] { failed_reassembly(true); }},
        {"level_shares_thin", [] { level_shares(320, 5, 5, 5); }},
        {"level_shares_deep", [] { level_shares(270, 15, 4, 4); }},
        {"level_shares_small", [] { level_shares(100, 4, 1, 1); }},
        {"one_product_per_solve", one_product},
        {"large_copies", [] { large_copies(false, false); }},
        {"large_copies_no_heap", [] { large_copies(true, false); }},
        {"large_copies_no_pinned", [] { large_copies(false, true); }},
        {"zero_store_no_ice", [] { zero_store(3, true); }},
        {"zero_store_outflow", [] { zero_store(1, false); }},
    };
    const auto c = checks.find(argv[2]);
    if (c == checks.end()) { printf("no check %s\n", argv[2]); return 2; }
    c->second();
    fflush(stdout);
    _Exit(bad ? 1 : 0);
}
