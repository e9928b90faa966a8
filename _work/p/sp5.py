W=[]
for n in (1,2,4,8,10): 
    for L in (16,100,250,400,600): run('%dx%d'%(n,L),32,8,128,[L]*n,256,None,W); run('%dx%d'%(n,L),32,8,128,[L]*n,0,None,W); run('%dx%d'%(n,L),16,4,128,[L]*n,0,dict(window=512),W)
for n in (11,14,16):
    for L in (16,300,700,760,1000,1500,4000,9000):
        run('%dx%d'%(n,L),32,8,128,[L]*n,0,None,W); run('%dx%d'%(n,L),32,8,128,[L]*n,1024,None,W)
    for a,b in ((100,6000),(1000,20000),(16,1000)): run('%dx%d-%d'%(n,a,b),32,8,128,logs(n,a,b),0,None,W); run('%dx%d-%d'%(2*n,a,b),28,4,128,logs(2*n,a,b),0,None,W)
for n in (8,12,16,21):
    for L in (16,600,650,1200,1300,2000): run('%dx%d'%(n,L),12,12,64,[L]*n,0,None,W); run('%dx%d'%(n,L),12,12,64,[L]*n,512,None,W)
    run('%dx100-2000'%n,12,12,64,logs(n,100,2000),0,None,W); run('%dx16-800'%n,12,12,64,logs(n,16,800),0,None,W)
for n in (40,64,90):
    run('%dx100-8000'%n,32,8,128,logs(n,100,8000),0,None,W)
    run('%dx100-8000 cap'%n,16,4,128,logs(n,100,8000),0,dict(cap=50.),W)
    run('%dx100-8000 win'%n,16,4,128,logs(n,100,8000),0,dict(window=1024),W)
    run('%dx300 cap'%n,32,8,128,[300]*n,0,dict(cap=50.),W)
