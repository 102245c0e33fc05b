// Emulate the matrix-core gradient kernel (felizjueves_amd/csrc/fj_gfquad.h)
// on the CPU over the launches of a gradient stream read from a binary file
// (the format of gfloop_emu.cpp); writes G. 256 threads, one per lane, one
// workgroup at a time. TEST INFRASTRUCTURE.
#include "fj_device.h"   // the emulation header, copied under this name
#include GFLOOP_HEADER
#include GFQUAD_HEADER
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

int main(int argc, char** argv) {
    std::ifstream f(argv[1], std::ios::binary);
    int n_launch, n_atom, n_ao;
    f.read((char*)&n_launch, 4);
    f.read((char*)&n_atom, 4);
    f.read((char*)&n_ao, 4);
    double* D = rd<double>(f);
    double* G = (double*)calloc((size_t)n_atom * 3 + 1, sizeof(double));
    struct L { FjGfArgs g; long long n; };
    std::vector<L> Ls(n_launch);
    for (auto& l : Ls) {
        int h[12];   // la lb lc ld n_bra n_ket k_ab k_cd n_atom n_ao diag chunk
        f.read((char*)h, sizeof h);
        double* bp = rd<double>(f); double* AB = rd<double>(f);
        int* bs = rd<int>(f); int* bao = rd<int>(f); int* bat = rd<int>(f);
        double* kp = rd<double>(f); double* CD = rd<double>(f);
        int* ks = rd<int>(f); int* kao = rd<int>(f); int* kat = rd<int>(f);
        l.g = FjGfArgs{h[0], h[1], h[2], h[3], h[4], h[5], h[6], h[7], h[8], h[9], h[10], h[11],
                       bp, AB, bs, bao, bat, kp, CD, ks, kao, kat, D, G};
        l.n = h[10] ? (long long)h[4] * (h[4] + 1) / 2 : (long long)h[4] * h[5];
        l.n *= (h[6] * h[7] + h[11] - 1) / h[11];
    }
    std::barrier<> bar(256), w0(64), w1(64), w2(64), w3(64);
    g_bar = &bar;
    g_wbar[0] = &w0; g_wbar[1] = &w1; g_wbar[2] = &w2; g_wbar[3] = &w3;
    blockDim = {256, 1, 1};
    std::vector<std::thread> ts;
    for (unsigned t = 0; t < 256; ++t)
        ts.emplace_back([&, t] {
            threadIdx = {t, 0, 0};
            for (auto& l : Ls) {
                const unsigned grid = (unsigned)std::min<long long>(l.n, 3);
                for (unsigned b = 0; b < grid; ++b) {
                    if (t == 0) { blockIdx = {b, 0, 0}; gridDim = {grid, 1, 1}; }
                    bar.arrive_and_wait();
                    switch (l.g.la * 1000 + l.g.lb * 100 + l.g.lc * 10 + l.g.ld) {
#define FJ_GQ_CLASS(a, b, c, d) \
    case a * 1000 + b * 100 + c * 10 + d: fj_gfquad_k<a, b, c, d>(l.g, nullptr, 0, l.n); break;
                        CLASSES
                        default: abort();
                    }
                    bar.arrive_and_wait();
                }
            }
        });
    for (auto& t : ts) t.join();
    std::ofstream out(argv[2], std::ios::binary);
    out.write((char*)G, 8LL * n_atom * 3);
    return 0;
}
