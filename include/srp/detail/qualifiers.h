/* Qualifier macros shared by the public headers.
 *
 * The public API is plain C.  The same headers are also read by HIP shader
 * modules (C++ compiled by hipcc), which need C linkage for the library entry
 * points and host+device definitions of the small math helpers that shaders
 * call. */
#pragma once

#ifdef __cplusplus
#  define SRP_EXTERN_C_BEGIN extern "C" {
#  define SRP_EXTERN_C_END }
#  define SRP_RESTRICT __restrict__
#else
#  define SRP_EXTERN_C_BEGIN
#  define SRP_EXTERN_C_END
#  define SRP_RESTRICT restrict
#endif

#if defined(__HIPCC__)
#  define SRP_HD __host__ __device__
#else
#  define SRP_HD
#endif

/* Shader modules compiled by hipcc get header-only host+device math.  The
 * library's own C translation unit that exports the math symbols defines
 * SRP_NO_INLINE_MATH. */
#if defined(__HIPCC__) && !defined(SRP_NO_INLINE_MATH)
#  define SRP_INLINE_MATH 1
#else
#  define SRP_INLINE_MATH 0
#endif

/* Device code: a generic pointer known to point to global memory, and one
 * to global memory that nothing writes while the kernel runs.  A pointer
 * read from memory has no known address space: loads through it are flat
 * (and wait for LDS traffic too), and a wave-uniform load that some store of
 * the kernel might alias goes through the vector memory path, several
 * hundred cycles each, instead of the scalar cache.  Casting to the address
 * space and back tells the compiler (by way of an integer: a direct pair of
 * casts is folded away); the pointer itself is unchanged. */
#if defined(__HIPCC__)
#include <stdint.h>
template <class T>
__host__ __device__ inline __attribute__((always_inline)) T* srpGlobal(T* p)
{
#if defined(__HIP_DEVICE_COMPILE__)
	return (T*) (__attribute__((address_space(1))) T*) (uintptr_t) p;
#else
	return p;
#endif
}
template <class T>
__host__ __device__ inline __attribute__((always_inline)) const T* srpConst(const T* p)
{
#if defined(__HIP_DEVICE_COMPILE__)
	return (const T*) (const __attribute__((address_space(4))) T*) (uintptr_t) p;
#else
	return p;
#endif
}
#endif
