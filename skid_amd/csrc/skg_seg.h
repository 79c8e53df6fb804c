// skg_seg.h -- segments of the members sorted by (group, iOrder).  Plain C++
// without device functions, so that a test can compile it for the host.
#pragma once
#ifndef SKG_SEG_FN
#define SKG_SEG_FN __device__ __forceinline__
#endif

// Where group g's members start: the first of the n sorted keys (group in the
// high 32 bits) that is not below g.  A group without members starts where the
// next one does, so the starts ascend with the id whatever ids are missing, and
// group g ends where g + 1 starts.
SKG_SEG_FN int group_start(const unsigned long long *key, int n, int g) {
	const unsigned long long k = (unsigned long long)(unsigned)g << 32;
	int lo = 0, hi = n;
	while (lo < hi) {
		const int mid = lo + ((hi - lo) >> 1);
		if (key[mid] < k) lo = mid + 1;
		else hi = mid;
	}
	return lo;
}

// The group >= 1 whose segment holds position t, 0 for none: the last group that
// starts at or before t (the starts ascend).
SKG_SEG_FN int group_at(const int *gs, const int *ge, int nG, int t) {
	int lo = 1, hi = nG - 1;
	while (lo < hi) {
		const int mid = lo + ((hi - lo + 1) >> 1);
		if (gs[mid] <= t) lo = mid;
		else hi = mid - 1;
	}
	return lo < nG && t >= gs[lo] && t < ge[lo] ? lo : 0;
}
