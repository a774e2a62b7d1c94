// Stand-ins for what hipcc's host code registers at start-up, so that a source file of the library compiles into
// a CPU program (--offload-host-only: no device code in it).
#pragma once
#include <stddef.h>

extern "C" {
void **__hipRegisterFatBinary(const void *) {
    static void *handle;
    return &handle;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *, void *, void *, int *) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
}
