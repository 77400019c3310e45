/* Stand-ins for the HIP runtime calls a launch makes, preloaded over the real
 * ones where there is no device: they count the launches and the limits
 * raised, and fail the raising of a kernel's LDS limit on demand. */
#include <stdlib.h>

typedef struct { unsigned x, y, z; } dim3_t;

static int last, launches, raised, fail, device;
static struct { dim3_t grid, block; size_t lds; void* stream; } call;

void stub_set(int fail_attribute, int current_device) { fail = fail_attribute; device = current_device; launches = raised = 0; }
int stub_launches(void) { return launches; }
int stub_raised(void) { return raised; }

int hipGetDevice(int* d) { *d = device; return 0; }
int hipGetLastError(void) { const int e = last; last = 0; return e; }
int hipFuncSetAttribute(const void* f, int attr, int value) {
    (void)f; (void)attr; (void)value;
    raised++;
    return fail ? (last = 1) : 0;
}
int __hipPushCallConfiguration(dim3_t g, dim3_t b, size_t lds, void* stream) {
    call.grid = g; call.block = b; call.lds = lds; call.stream = stream;
    return 0;
}
int __hipPopCallConfiguration(dim3_t* g, dim3_t* b, size_t* lds, void** stream) {
    *g = call.grid; *b = call.block; *lds = call.lds; *stream = call.stream;
    return 0;
}
int hipLaunchKernel(const void* f, dim3_t g, dim3_t b, void** args, size_t lds, void* stream) {
    (void)f; (void)g; (void)b; (void)args; (void)lds; (void)stream;
    launches++;
    return 0;
}
