from .manager import BatchArrays, CacheError, CacheGroup, DecodeStepError, OutOfPages, PagedCacheManager, busiest_over_share
