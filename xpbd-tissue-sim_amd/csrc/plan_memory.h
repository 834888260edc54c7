// Device memory of a plan: all its lists and arrays in one allocation, and its small
// lists in one copy.  An allocation or a copy is some 10 us, and a plan has fifteen to
// fifty arrays: 4^3 cells 280 us for the plan, now 50.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstring>
#include <vector>

#include "capi_internal.h"

namespace xpbd {

class PlanMemory {
public:
    // *dst: a device copy of v, which has to stay until place()
    template <typename D, typename T>
    void put(const D** dst, const std::vector<T>& v)
    {
        static_assert(sizeof(D) % sizeof(T) == 0, "D is made of Ts");
        add(lists_, reinterpret_cast<void**>(const_cast<D**>(dst)), v.data(), sizeof(T) * v.size());
    }
    // *dst: n zeros
    template <typename T>
    void zeros(T** dst, size_t n)
    {
        add(zeros_, reinterpret_cast<void**>(dst), nullptr, sizeof(T) * n);
    }
    // *dst: room for n
    template <typename T>
    void room(T** dst, size_t n)
    {
        add(rooms_, reinterpret_cast<void**>(dst), nullptr, sizeof(T) * n);
    }

    // Allocates, copies, and enqueues the zeros' fill.
    int place(xpbd_handle* h)
    {
        size_t at = 0;
        for (Array& a : lists_)
            if (a.bytes <= kSmall) a.at = at, at += round(a.bytes);
        std::vector<char> small(at);   // the small lists, as they will lie
        const size_t sent = at;
        for (Array& a : lists_) {
            if (a.bytes > kSmall) a.at = at, at += round(a.bytes);
            else if (a.bytes) std::memcpy(small.data() + a.at, a.from, a.bytes);
        }
        const size_t zero = at;
        for (Array& a : zeros_) a.at = at, at += round(a.bytes);
        const size_t rest = at;
        for (Array& a : rooms_) a.at = at, at += round(a.bytes);
        void* p = nullptr;
        int rc = dalloc_bytes(h, &p, at);
        if (rc) return rc;
        char* const base = static_cast<char*>(p);
        hipError_t e = sent ? hipMemcpy(base, small.data(), sent, hipMemcpyHostToDevice) : hipSuccess;
        for (const Array& a : lists_)
            if (e == hipSuccess && a.bytes > kSmall) e = hipMemcpy(base + a.at, a.from, a.bytes, hipMemcpyHostToDevice);
        if (e == hipSuccess && rest > zero) e = launch_fill_zero(h->stream, base + zero, rest - zero);
        if (e != hipSuccess) return hip_err(h, e, "plan memory");
        for (const auto* part : { &lists_, &zeros_, &rooms_ })
            for (const Array& a : *part) *a.dst = base + a.at;
        return XPBD_OK;
    }

private:
    static constexpr size_t kSmall = 64 * 1024;   // longer ones are not worth a second copy on the host
    static size_t round(size_t n) { return (n + 255) / 256 * 256; }
    struct Array {
        void** dst;
        const void* from;
        size_t bytes, at;
    };
    void add(std::vector<Array>& part, void** dst, const void* from, size_t bytes) { part.push_back({ dst, from, bytes, 0 }); }
    std::vector<Array> lists_, zeros_, rooms_;
};

}  // namespace xpbd
