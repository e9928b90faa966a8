def old(T,n,G,kv,K):
    w=(T*G//256+n)*kv
    return w>=440 and K>=2048 and T>=256*n and (w<=1100 or T>=1024*n)
def new(T,n,G,kv,K):
    each=(T*G+n*256-1)//(n*256)
    w=each*n*kv
    if w<440 or K<2048 or T<256*n: return False
    if w<=512: return True
    if w<=640 or K<3072: return False
    if w>1100 and T<1024*n: return False
    return n>1 or 2*K>=3*T or K>=6144
def case(lens,ctx,kv,per):
    import math
    K=max(a+b for a,b in zip(lens,ctx)); K=(K+15)//16*16
    T,n=sum(lens),len(lens)
    print(lens if n<9 else n,ctx if n<9 else '',kv,per,'w',(-(-T*per//(n*256)))*n*kv,'wgs',(T*per//256+n)*kv,'K',K,old(T,n,per,kv,K),new(T,n,per,kv,K))
if __name__=='__main__':
    for c in [([900,1,257,32,0,433],[0,2300,17,5,9,100],16,8),([700,333],[0,2100],15,7),([600,500],[1500,0],32,3),([1100],[950],88,1),([260]*65+[300],[0]*65+[1800],4,2),
      ([900,300,5],[450-900,0,2300-5],16,8),([900],[1300],16,8),([610,500],[40,1600],32,3),([4096],[0],8,4),([2000],[0],32,1),
      ([900, 700], [0, 1200], 16, 8)]: case(*c)
