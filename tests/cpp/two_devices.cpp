// bf16n_init with one and with another device current, against HIP calls that only count: prints, per device, the kernels whose
// shared-memory limit was raised there and the look-ups of the routing lists' address.  Runs without a GPU.
#include <bf16n_c.h>

#include <cstdio>
#include <set>

static int device = 0, symbols[2];
static std::set<const void *> raised[2];

extern "C" {
int hipGetDevice(int * d) { *d = device; return 0; }
int hipDeviceGetAttribute(int * v, int, int) { *v = 256; return 0; }
int hipFuncSetAttribute(const void * f, int, int) { raised[device].insert(f); return 0; }
int hipGetSymbolAddress(void ** p, const void *) { symbols[device]++; *p = &symbols[device]; return 0; }
}

int main() {
    for (int d : {0, 1, 0, 1}) {
        device = d;
        if (bf16n_init() != 0) {
            std::printf("error %s\n", bf16n_last_error());
            return 1;
        }
    }
    std::printf("%zu %d %zu %d %d\n", raised[0].size(), symbols[0], raised[1].size(), symbols[1], (int) (raised[0] == raised[1]));
    return 0;
}
