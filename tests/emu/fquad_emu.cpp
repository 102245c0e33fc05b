// Emulate the matrix-core F kernel (felizjueves_amd/csrc/fj_fquad.h) on the
// CPU over walker launches read from a binary file (the format of
// floop_emu.cpp); writes F. 256 threads, one per lane, one workgroup at a
// time. CLASSES: FJ_FQ_CLASS(la, lb, lc, ld) of each class in the file.
// TEST INFRASTRUCTURE.
#include "fj_device.h"   // the emulation header, copied under this name
#include FQUAD_HEADER
#include <fstream>
#include <thread>
#include <vector>
thread_local uint3e threadIdx;
uint3e blockIdx, blockDim, gridDim;
std::barrier<>* g_bar;
std::barrier<>* g_wbar[4];
double g_mfa[2][256], g_mfb[2][256];
thread_local int g_mf_parity;
double g_shfl[256];
double* g_dyn_lds;

template <typename T> T* rd(std::ifstream& f) {
    long long n;
    f.read((char*)&n, 8);
    T* p = (T*)malloc(n * sizeof(T) + 1);   // exactly sized, so ASan sees an overrun
    f.read((char*)p, n * sizeof(T));
    return p;
}

// a class's workgroup, or (a null) its number of workgroups to a ket
static int run(const int* c, int span, const FjFArgs* a) {
#define FJ_FQ_CLASS(A, B, C, D) \
    if (c[0] == A && c[1] == B && c[2] == C && c[3] == D) { \
        if (a) fj_fquad_k<A, B, C, D>(span, *a); \
        return Fq<A, B, C, D>::Z; \
    }
    CLASSES
    return 0;
}

int main(int argc, char** argv) {
    std::ifstream f(argv[1], std::ios::binary);
    int hdr[2];   // n_launch n_ao
    f.read((char*)hdr, sizeof hdr);
    const int n_ao = hdr[1], span = 64;
    struct L { int c[4]; FjFArgs a; };
    std::vector<L> Ls(hdr[0]);
    double* F = (double*)calloc((size_t)n_ao * n_ao, 8);
    for (auto& l : Ls) {
        int h[11];   // la lb lc ld n_bra n_ket k_ab k_cd n_sh n_ao diag
        f.read((char*)h, sizeof h);
        double tau;
        f.read((char*)&tau, 8);
        for (int i = 0; i < 4; ++i) l.c[i] = h[i];
        double* bp = rd<double>(f); double* AB = h[1] ? rd<double>(f) : nullptr;
        double* Gab = rd<double>(f); int* bsh = rd<int>(f); int* bao = rd<int>(f);
        double* kp = rd<double>(f); double* CD = h[3] ? rd<double>(f) : nullptr;
        double* Gcd = rd<double>(f); int* ksh = rd<int>(f); int* kao = rd<int>(f);
        double* Dsh = rd<double>(f); double* D = rd<double>(f);
        FjFArgs& a = l.a;
        a.bra = FjSide{bp, nullptr, h[6], AB, Gab, bsh, bao, h[4]};
        a.ket = FjSide{kp, nullptr, h[7], CD, Gcd, ksh, kao, h[5]};
        a.work = nullptr; a.ket_list = nullptr; a.sys = nullptr;
        a.one = FjSys{D, Dsh, F, n_ao, h[8]};
        a.diag = h[10]; a.tau = tau;
        a.ws = nullptr; a.ws_doubles = 0; a.n_fp64 = 0; a.tier = nullptr; a.n_bx = 0; a.n_items = 0;
    }
    std::barrier<> bar(256), w0(64), w1(64), w2(64), w3(64);
    g_bar = &bar;
    g_wbar[0] = &w0; g_wbar[1] = &w1; g_wbar[2] = &w2; g_wbar[3] = &w3;
    blockDim = {256, 1, 1};
    std::atomic<bool> ok{true};
    std::vector<std::thread> ts;
    for (unsigned t = 0; t < 256; ++t)
        ts.emplace_back([&, t] {
            threadIdx = {t, 0, 0};
            for (auto& l : Ls) {
                const unsigned gx = l.a.bra.n, gy = (l.a.ket.n + span - 1) / span, gz = run(l.c, span, nullptr);
                if (!gz) ok = false;
                for (unsigned z = 0; z < gz; ++z)
                    for (unsigned y = 0; y < gy; ++y)
                        for (unsigned x = 0; x < gx; ++x) {
                            if (t == 0) { blockIdx = {x, y, z}; gridDim = {gx, gy, gz}; }
                            bar.arrive_and_wait();
                            run(l.c, span, &l.a);
                            bar.arrive_and_wait();
                        }
            }
        });
    for (auto& t : ts) t.join();
    std::ofstream o(argv[2], std::ios::binary);
    o.write((char*)F, 8LL * n_ao * n_ao);
    return ok ? 0 : 1;
}
