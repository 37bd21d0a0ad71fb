// staging.cpp -- small transfers through page-locked memory (bem_internal.h).
#include <cstring>

#include "bem_internal.h"

namespace {

bool pin_ready(bem_ctx* c) {
    if (!c->pin && !c->pin_tried) {
        c->pin_tried = true;
        void* p = nullptr;
        if (hipHostMalloc(&p, kPinBytes, hipHostMallocDefault) == hipSuccess)
            c->pin = static_cast<char*>(p);
        else
            (void)hipGetLastError();
    }
    return c->pin != nullptr;
}

size_t pin_round(size_t bytes) { return (bytes + 63) / 64 * 64; }

}  // namespace

int ctx_put(bem_ctx* c, void* dst, const void* src, size_t bytes) {
    if (bytes > kPinBytes / 2 || !pin_ready(c)) {
        BEM_HIP(c, hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, c->stream));
        BEM_HIP(c, hipStreamSynchronize(c->stream));  // the caller's memory is its own again
        return 0;
    }
    if (c->pin_off + bytes > kPinBytes) {
        BEM_HIP(c, hipStreamSynchronize(c->stream));
        c->pin_off = 0;
    }
    char* p = c->pin + c->pin_off;
    std::memcpy(p, src, bytes);
    c->pin_off += pin_round(bytes);
    BEM_HIP(c, hipMemcpyAsync(dst, p, bytes, hipMemcpyHostToDevice, c->stream));
    return 0;
}

int ctx_fetch(bem_ctx* c, std::initializer_list<Fetch> list) {
    const size_t start = c->pin_off;
    size_t off = start;
    // the same walk twice: queue the copies, then move the staged ones out
    for (const Fetch& f : list) {
        void* to = f.dst;
        if (off + f.bytes <= kPinBytes && pin_ready(c)) {
            to = c->pin + off;
            off += pin_round(f.bytes);
        }
        BEM_HIP(c, hipMemcpyAsync(to, f.src, f.bytes, hipMemcpyDeviceToHost, c->stream));
    }
    BEM_HIP(c, hipStreamSynchronize(c->stream));
    off = start;
    for (const Fetch& f : list)
        if (off + f.bytes <= kPinBytes && c->pin) {
            std::memcpy(f.dst, c->pin + off, f.bytes);
            off += pin_round(f.bytes);
        }
    c->pin_off = 0;
    return 0;
}
