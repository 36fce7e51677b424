// Stands in for the HIP runtime's launch calls so that the library's dispatch can be checked
// without a GPU: every launch is noted (kernel name, grid, block, LDS) and
// reported as successful. Loaded with RTLD_GLOBAL ahead of the library.
#include <cstddef>
#include <cstdint>
#include <map>
#include <string>
#include <vector>

struct Dim3 {
    uint32_t x, y, z;
};

struct Launch {
    const char * name;
    uint32_t     grid[3];
    uint32_t     block[3];
    uint64_t     lds;
};

struct Config {
    Dim3   grid, block;
    size_t lds;
    void * stream;
};

static Config & config() {
    static Config c;
    return c;
}

static std::map<const void *, std::string> & names() {
    static std::map<const void *, std::string> m;
    return m;
}

static std::vector<Launch> & launches() {
    static std::vector<Launch> v;
    return v;
}

extern "C" {

// (not passed on: nothing is launched)
void __hipRegisterFunction(void **, const void * host, char *, const char * name, unsigned, void *, void *, void *, void *, int *) {
    names()[host] = name;
}

int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t lds, void * stream) {
    config() = { grid, block, lds, stream };
    return 0;
}

int __hipPopCallConfiguration(Dim3 * grid, Dim3 * block, size_t * lds, void ** stream) {
    *grid   = config().grid;
    *block  = config().block;
    *lds    = config().lds;
    *stream = config().stream;
    return 0;
}

int hipLaunchKernel(const void * f, Dim3 grid, Dim3 block, void **, size_t lds, void *) {
    launches().push_back(Launch{ names()[f].c_str(), { grid.x, grid.y, grid.z }, { block.x, block.y, block.z }, lds });
    return 0;
}

int hipGetLastError() {
    return 0;
}

int launch_count() {
    return static_cast<int>(launches().size());
}

const Launch * launch_at(int i) {
    return &launches()[static_cast<size_t>(i)];
}

void launch_clear() {
    launches().clear();
}
}
