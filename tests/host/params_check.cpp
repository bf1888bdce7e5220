// A kernel's parameters declared without braces (`LinearF32Params p;`) are those of `LinearF32Params{}`: no pointer, count or factor keeps what the memory held before.  ALL_PARAMS: every
// struct of that kind in the kernels' headers, as CHECK(name) one after the other.  No device, no library.
#include <cstdio>
#include <cstring>
#include <new>

#include "../../uzu_amd/csrc/kernels.h"
#include "../../uzu_amd/csrc/kernels_decode.h"
#include "../../uzu_amd/csrc/kernels_stream32.h"

using namespace uzu::k;

// the bytes of both, padding cleared, over memory full of ones (the barriers keep the fill, which the compiler may drop in front of an object's beginning)
template <class T> int check(const char* name) {
    alignas(T) static unsigned char plain[sizeof(T)], braces[sizeof(T)];
    memset(plain, 0xff, sizeof plain), memset(braces, 0xff, sizeof braces);
    asm volatile("" ::: "memory");
    T* a = new (plain) T;
    T* b = new (braces) T{};
    asm volatile("" ::: "memory");
    __builtin_clear_padding(a), __builtin_clear_padding(b);
    const bool same = memcmp(plain, braces, sizeof plain) == 0;
    if (!same) printf("%s: undefined members without braces\n", name);
    return !same;
}

int main() {
    int bad = 0, structs = 0;
#define CHECK(name) bad += check<name>(#name), ++structs;
    ALL_PARAMS
    printf("%d structs\n%d bad\n", structs, bad);
    return bad != 0;
}
