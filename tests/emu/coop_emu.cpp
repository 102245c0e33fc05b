// Emulate an F kernel of one class over a builder work list read from a
// binary file; writes F: the quartet-cooperative one (gen/c_<cls>.h), or the
// call CALL of any other, with GRID_Z workgroups to each (x, y).
// 256 threads, one per lane, one workgroup at a time. TEST INFRASTRUCTURE.
#include "fj_device.h"   // the emulation header, copied under this name
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
#include CLS_HEADER
#ifndef CALL
#define CALL KERNEL<true>(a, parent, 2.0, -0.5)
#define GRID_Z 1
#endif

template <typename T> T* rd(std::ifstream& f) {
    long long n;
    f.read((char*)&n, 8);
    T* p = (T*)malloc(n * sizeof(T) + 1);   // exactly sized, so ASan sees an overrun
    f.read((char*)p, n * sizeof(T));
    return p;
}

int main(int argc, char** argv) {
    std::ifstream f(argv[1], std::ios::binary);
    int h[7];   // n_bra n_ket n_work parts n_sh n_ao diag
    f.read((char*)h, sizeof h);
    double tau;
    f.read((char*)&tau, 8);
    FjFArgs a;
    FjSide* sides[2] = {&a.bra, &a.ket};
    for (int i = 0; i < 2; ++i) {
        double* prim = rd<double>(f); int* off = rd<int>(f); double* sep = rd<double>(f);
        double* G = rd<double>(f); int* sh = rd<int>(f); int* ao = rd<int>(f);
        *sides[i] = FjSide{prim, off, 0, sep, G, sh, ao, h[i]};
    }
    a.work = (const int4*)rd<int>(f);
    a.ket_list = rd<int>(f);
    const int* parent = rd<int>(f);
    a.tier = rd<int>(f);
    double* Dsh = rd<double>(f); double* D = rd<double>(f);
    double* F = (double*)calloc((size_t)h[5] * h[5], 8);
    FjSys sys{D, Dsh, F, h[5], h[4]};
    a.sys = &sys; a.one = sys; a.diag = h[6]; a.tau = tau;
    a.ws = nullptr; a.ws_doubles = 0; a.n_bx = h[2]; a.n_items = h[2]; a.n_fp64 = 0;
    std::barrier<> bar(256), w0(64), w1(64), w2(64), w3(64);
    g_bar = &bar;
    g_wbar[0] = &w0; g_wbar[1] = &w1; g_wbar[2] = &w2; g_wbar[3] = &w3;
    blockDim = {256, 1, 1};
    gridDim = {(unsigned)h[2], (unsigned)h[3], GRID_Z};
    std::vector<std::thread> ts;
    for (unsigned t = 0; t < 256; ++t)
        ts.emplace_back([&, t] {
            threadIdx = {t, 0, 0};
            for (unsigned z = 0; z < gridDim.z; ++z)
                for (unsigned y = 0; y < gridDim.y; ++y)
                    for (unsigned x = 0; x < gridDim.x; ++x) {
                        if (t == 0) blockIdx = {x, y, z};
                        bar.arrive_and_wait();
                        CALL;
                        bar.arrive_and_wait();
                    }
        });
    for (auto& t : ts) t.join();
    std::ofstream o(argv[2], std::ios::binary);
    o.write((char*)F, 8LL * h[5] * h[5]);
    return 0;
}
